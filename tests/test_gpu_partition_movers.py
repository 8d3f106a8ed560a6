"""GPU parity of the hint partition's mover ordering where it can go wrong: a
cell at, below and above the mover count from which a workgroup orders it, and
the remainders of the workgroups (particles per classify block, per word of
stay bits, cells per scan thread). Bar: bit-exact against numpy's stable
argsort of the cell keys (thrust::stable_sort_by_key,
spatialpartition.cpp:113-117), for an unsorted hint (every particle a mover)
and for a sorted one with few movers."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _run(ctx, g, keys_to_x, keys, hint):
    from pyroclastmpm_amd import capi
    n, dev = len(keys), torch.device("cuda")
    x = torch.from_numpy(np.ascontiguousarray(keys_to_x(keys).T)).to(dev)
    hs = torch.from_numpy(hint.astype(np.uint32).view(np.int32).copy()).to(dev)
    h, so = torch.zeros(n, dtype=torch.int32, device=dev), torch.full((n,), -1, dtype=torch.int32, device=dev)
    cs, ce = (torch.full((g.num_cells_total,), 7, dtype=torch.int32, device=dev) for _ in range(2))
    sp = capi.Spatial(h.data_ptr(), hs.data_ptr(), so.data_ptr(), cs.data_ptr(), ce.data_ptr(), None)
    capi.check(capi.lib().pmpm_partition(ctx.ptr, 2, C.byref(g), x.data_ptr(), n, C.byref(sp),
                                         torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return so.cpu().numpy(), hs.cpu().numpy(), cs.cpu().numpy(), ce.cpu().numpy()


@pytest.mark.parametrize("big", [1, 2047, 2048, 2049, 9001])
@pytest.mark.parametrize("rest", [1, 255, 1027])
def test_mover_order_at_the_edges(big, rest):
    from pyroclastmpm_amd import capi
    nx, ny, hcell = 37, 29, 0.5
    g = capi.make_grid([0, 0, 0], [(nx - 0.75) * hcell, (ny - 0.75) * hcell, 0], hcell, 2)
    assert g.num_cells_total == nx * ny
    rng = np.random.default_rng(big * 7 + rest)
    keys = np.concatenate([np.full(big, 400), np.full(big // 2 + 3, 77), rng.integers(0, nx * ny, rest)])
    rng.shuffle(keys)
    to_x = lambda k: np.stack([(k % nx + 0.5) * hcell, (k // nx + 0.5) * hcell], axis=1).astype(np.float32)
    ctx = capi.Context(len(keys), g.num_cells_total)
    prev = np.sort(keys)
    moved = prev.copy()  # the sorted keys as hint, three of them changed since
    at = rng.integers(0, len(moved), 3)
    moved[at] = rng.integers(0, nx * ny, 3)
    for k, hint in ((keys, rng.integers(0, 2 ** 31, len(keys))), (moved, prev), (keys, np.zeros(len(keys), np.int64))):
        so, hs, cs, ce = _run(ctx, g, to_x, k, hint)
        order = np.argsort(k, kind="stable")
        np.testing.assert_array_equal(so, order)
        np.testing.assert_array_equal(hs, k[order])
        cnt = np.bincount(k, minlength=nx * ny)
        end = np.cumsum(cnt)
        np.testing.assert_array_equal(ce, np.where(cnt > 0, end, 0))
        np.testing.assert_array_equal(cs, np.where(cnt > 0, end - cnt, 0))
