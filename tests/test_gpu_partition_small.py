"""GPU parity of the one-workgroup partition of small scenes at its edges: the
particle counts where its layouts begin and end (and the first count past it),
no particle outside, some, all; every particle in one cell; a sorted input.
Bar: bit-exact against numpy's stable argsort of the cell keys
(thrust::stable_sort_by_key, spatialpartition.cpp:113-117)."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("n", [1, 2, 63, 511, 512, 513, 1024, 1025, 2047, 2048, 2049])
@pytest.mark.parametrize("cells", [(1,), (7, 5), (128, 128), (23, 27, 26), (129, 128)])
def test_small_partition(n, cells):
    from pyroclastmpm_amd import capi
    dim, h, dev = len(cells), 0.5, torch.device("cuda")
    g = capi.make_grid([0, 0, 0], [(c - 0.75) * h for c in cells] + [0] * (3 - dim), h, dim)
    nc = g.num_cells_total
    assert nc == int(np.prod(cells))
    rng = np.random.default_rng(n + nc)
    ctx = capi.Context(n, nc)
    stride = np.cumprod((1,) + cells[:-1])
    some = np.where(rng.random(n) < 0.1, nc, rng.integers(0, nc, n))
    for keys in (rng.integers(0, nc, n), some, np.sort(some), np.full(n, nc), np.full(n, nc - 1)):
        b = (keys[:, None] // stride) % np.array(cells)
        x = ((b + 0.5) * h).astype(np.float32)
        x[keys == nc] = 1e4  # past the last cell
        xs = torch.from_numpy(np.ascontiguousarray(x.T)).to(dev)
        i32 = lambda m, v: torch.full((m,), v, dtype=torch.int32, device=dev)
        ha, hs, so, bins = i32(n, -1), i32(n, 0), i32(n, -1), i32(dim * n, -1)
        cs, ce = i32(nc, 7), i32(nc, 7)
        sp = capi.Spatial(ha.data_ptr(), hs.data_ptr(), so.data_ptr(), cs.data_ptr(), ce.data_ptr(), bins.data_ptr())
        stream = torch.cuda.current_stream().cuda_stream
        capi.check(capi.lib().pmpm_partition(ctx.ptr, dim, C.byref(g), xs.data_ptr(), n, C.byref(sp), stream))
        out = C.c_int32(-1)
        capi.check(capi.lib().pmpm_context_out_of_grid(ctx.ptr, stream, C.byref(out)))
        torch.cuda.synchronize()
        order = np.argsort(keys, kind="stable")
        inside = np.bincount(keys[keys < nc], minlength=nc)
        end = np.cumsum(inside)
        np.testing.assert_array_equal(ha.cpu().numpy(), keys)
        np.testing.assert_array_equal(so.cpu().numpy(), order)
        np.testing.assert_array_equal(hs.cpu().numpy(), keys[order])
        np.testing.assert_array_equal(cs.cpu().numpy(), np.where(inside > 0, end - inside, 0))
        np.testing.assert_array_equal(ce.cpu().numpy(), np.where(inside > 0, end, 0))
        assert out.value == int((keys == nc).sum())
        np.testing.assert_array_equal(bins.cpu().numpy().reshape(dim, n).T[keys < nc], b[keys < nc])
