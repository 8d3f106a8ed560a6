"""GPU: the first partition of a reserved context is only recorded into a HIP
graph. The context's counts must be zero between calls, so an eager partition
that comes before the graph's first replay must find them cleared, and the
replays must too. Bar: bit-exact against numpy's stable argsort of the cell
keys (thrust::stable_sort_by_key, spatialpartition.cpp:113-117) for the eager
call and for every replay, with eager calls in between."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


# (one workgroup; classify, scan, movers, place)
@pytest.mark.parametrize("n", [700, 5000])
def test_first_partition_recorded_then_eager(n):
    from pyroclastmpm_amd import capi
    nx, ny, dev = 61, 47, torch.device("cuda")
    g = capi.make_grid([0, 0, 0], [nx - 0.75, ny - 0.75, 0], 1.0, 2)
    nc = g.num_cells_total
    rng = np.random.default_rng(n)
    # workspace freed by others holds anything: leave floats where the context's may come to lie
    junk = [torch.full((1 << 16,), 1e9, device=dev) for _ in range(8)]
    torch.cuda.synchronize()
    del junk
    torch.cuda.empty_cache()
    ctx = capi.Context(n, nc)
    x = torch.zeros((2, n), device=dev)
    t = {k: torch.zeros(m, dtype=torch.int32, device=dev)
         for k, m in (("hash", n), ("hash_sorted", n), ("sorted", n), ("cell_start", nc), ("cell_end", nc))}
    sp = capi.Spatial(*[t[k].data_ptr() for k in ("hash", "hash_sorted", "sorted", "cell_start", "cell_end")], None)

    def partition():
        capi.check(capi.lib().pmpm_partition(ctx.ptr, 2, C.byref(g), x.data_ptr(), n, C.byref(sp),
                                             torch.cuda.current_stream().cuda_stream))

    def positions():
        keys = rng.integers(0, nc, n)
        x.copy_(torch.from_numpy(np.stack([keys % nx + 0.5, keys // nx + 0.5]).astype(np.float32)))
        return keys

    def check(keys, what):
        torch.cuda.synchronize()
        order = np.argsort(keys, kind="stable")
        cnt = np.bincount(keys, minlength=nc)
        np.testing.assert_array_equal(t["sorted"].cpu().numpy(), order, err_msg=what)
        np.testing.assert_array_equal(t["hash_sorted"].cpu().numpy(), keys[order], err_msg=what)
        np.testing.assert_array_equal(t["cell_end"].cpu().numpy(), np.where(cnt > 0, np.cumsum(cnt), 0), err_msg=what)

    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        partition()
    keys = positions()
    partition()
    check(keys, "eager, before the first replay")
    for k in range(3):
        keys = positions()
        graph.replay()
        check(keys, f"replay {k}")
        keys = positions()
        partition()
        check(keys, f"eager after replay {k}")
