"""GPU: the recomputed steps of a checkpoint segment hand their sorted keys on,
so the next partition has them as its hint, and the gradient is the same to the
last bit as with a hint of each step's own (which only ever changes the time)."""
import numpy as np
import pytest

from tests import scenarios as S

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def test_recomputed_steps_hand_their_hint_on():
    from pyroclastmpm_amd.diff import DiffMPM, StepBuffers

    spec = S.column(h=0.04, per_axis=2, dt=1e-3, jitter=0.1, seed=2, musl=False)
    theta, steps, out = (28.0, 200.0, 1e5), 12, []
    for own in (False, True):
        m = DiffMPM(3, spec.origin, spec.end, 0.04, spec.positions, 8, dt=1e-3, checkpoint_every=5)
        assert m.n > 2048  # (fewer are sorted by one workgroup, without a hint)
        _, work = m._segment_buffers()
        if own:
            work[1:] = [StepBuffers(m.n, m.grid.num_cells_total, 3) for _ in work[1:]]
        else:
            assert len({w.sp["hash_sorted"].data_ptr() for w in work}) == 1
            assert all(w.spatial.hash_sorted == work[0].spatial.hash_sorted for w in work)
        final, ckpts = m.forward(theta, steps)
        gx = torch.from_numpy(np.random.default_rng(0).standard_normal((m.n, 3))).float().cuda()
        out.append(m.backward(theta, steps, ckpts, final, gx))
    assert np.array_equal(out[0], out[1]) and np.abs(out[0]).max() > 0
