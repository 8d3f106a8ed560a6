"""GPU: the 3D cubic adjoint step with sixteen lanes per particle in the adjoint
P2G (the layout of small launches) against the FP64 oracle's finite
differences, with the one-step check's bar (2e-3)."""
import pytest

from tests import test_gpu_adjoint as A

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def test_sixteen_lanes_match_fp64_oracle(oracle_mod, monkeypatch):
    monkeypatch.setenv("PMPM_ADJOINT_P2G_LANES", "16")
    pos, geo = A._column_3d(h=0.05, per_axis=3)
    A._one_step_check(oracle_mod, pos, geo, label="lanes 16")
