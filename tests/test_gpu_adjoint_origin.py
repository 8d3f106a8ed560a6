"""GPU: the adjoint step of a column whose first particles lie left of the
origin (coordinates in (-1, 0) cells: truncated to cell 0, negative fraction).
The forward step deposits and gathers them (usl_inline.h:104-160, 262-305), so
the adjoint scatter has to hand their G2P adjoints to the nodes too. Bar: that
of the one-step check (2e-3) against the FP64 oracle's finite differences, with
the loss on the particles near the origin, where such a particle's share is
large."""
import numpy as np
import pytest

from tests import test_gpu_adjoint as A

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("dim", [2, 3])
def test_one_step_adjoint_left_of_the_origin(oracle_mod, dim):
    h = 0.05
    pos, geo = A._column_2d(h=h) if dim == 2 else A._column_3d(h=h, per_axis=3)
    pos = np.array(pos)
    pos[:, 0] -= 0.5 * h  # the first layer of particles: t from about -0.4 to 0
    print(f"\n[gpu-test] {dim}D, {int((pos[:, 0] < 0).sum())} of {len(pos)} particles left of the origin", flush=True)
    left = []

    def keep(x):
        left.append(int((x[0] < 0).sum()))
        return x[0] < 0.6 * h

    A._one_step_check(oracle_mod, pos, geo, label="left of the origin", keep=keep)
    assert left[0] > 0.08 * len(pos), "the state must still have such particles"
