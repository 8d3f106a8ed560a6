"""GPU: a 3D particle with a field that is not finite spoils the nodes of its
own window and no others, in the P2G and in the MUSL re-map, whatever the
spline and the tiles (small scenes and larger ones take different ones). The
matrix products form four node offsets per axis; the linear spline has two."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("n", [900, 17000])
@pytest.mark.parametrize("sf, lo, hi", [("linear", 0, 1), ("quadratic", -1, 2), ("cubic", -1, 2)])
def test_nonfinite_fields_stay_in_the_window(sf, lo, hi, n):
    from pyroclastmpm_amd import capi
    dev, cells = torch.device("cuda"), (19, 9, 11)
    g = capi.make_grid([0, 0, 0], [c - 0.75 for c in cells], 1.0, 3)
    nn = g.num_cells_total
    rng = np.random.default_rng(n)
    pos = (rng.uniform(0.0, 1.0, (n, 3)) * (np.array(cells) - 4.0) + 1.5).astype(np.float32)
    bad = n // 2
    pos[bad] = [8.3, 4.6, 5.4]
    f = lambda *s: torch.zeros(*s, device=dev)
    i32 = lambda m: torch.zeros(m, dtype=torch.int32, device=dev)

    def particles():
        t = {"x": f(3, n), "v": f(3, n), "stress": f(6, n), "F": f(9, n), "L": f(9, n), "mass": f(n) + 1, "volume": f(n) + 0.1,
             "volume0": f(n) + 0.1, "color": torch.zeros(n, dtype=torch.uint8, device=dev),
             "flags": torch.full((n,), capi.PF_ACTIVE, dtype=torch.uint8, device=dev), "id": i32(n)}
        t["x"].copy_(torch.from_numpy(np.ascontiguousarray(pos.T)))
        t["v"].copy_(torch.from_numpy(rng.normal(size=(3, n)).astype(np.float32)))
        t["stress"].copy_(torch.from_numpy(rng.normal(size=(6, n)).astype(np.float32)))
        return t, capi.Particles(n, *[t[k].data_ptr() for k in ["x", "v", "stress", "F", "L", "mass", "volume", "volume0",
                                                                "color", "flags", "id"]])

    (a, pa), (b, pb) = particles(), particles()
    sp = {"hash": i32(n), "hash_sorted": i32(n), "sorted": i32(n), "cell_start": i32(nn), "cell_end": i32(nn)}
    part = capi.Spatial(*[sp[k].data_ptr() for k in sp], None)
    nd = {"mass": f(nn), "mom": f(3 * nn), "mom_nt": f(3 * nn), "vel": f(8 * nn)}
    nodes = capi.Nodes(*[nd[k].data_ptr() for k in nd])
    prm = capi.Params()
    prm.dim, prm.shape_fn, prm.dt, prm.alpha = 3, capi.SF[sf], 1e-3, 0.99
    prm.small_mass_cutoff, prm.node_types_built, prm.wrap_quirk = 1e-9, int(sf == "cubic"), 1
    ctx, L, s = capi.Context(n, nn), capi.lib(), torch.cuda.current_stream().cuda_stream
    k = np.arange(nn)
    ids = np.stack([k % cells[0], (k // cells[0]) % cells[1], k // (cells[0] * cells[1])], 1)
    cell = np.floor(pos[bad]).astype(int)
    window = np.all((ids >= cell + lo) & (ids <= cell + hi), axis=1)

    def spoilt():
        torch.cuda.synchronize()
        return ~np.isfinite(nd["mom_nt"].cpu().numpy().reshape(3, nn)).all(axis=0)

    for value in (float("inf"), float("nan")):
        a["stress"][0, bad] = value
        capi.check(L.pmpm_partition(ctx.ptr, 3, C.byref(g), a["x"].data_ptr(), n, C.byref(part), s))
        capi.check(L.pmpm_p2g(ctx.ptr, C.byref(prm), C.byref(g), C.byref(pa), C.byref(part), C.byref(nodes), s))
        bad_nodes = spoilt()
        assert bad_nodes.any() and not (bad_nodes & ~window).any(), (value, np.nonzero(bad_nodes & ~window)[0])
        a["stress"][0, bad] = 0.0
        # the re-map deposits m v' of the first map: a velocity that is not finite reaches it alone
        capi.check(L.pmpm_p2g(ctx.ptr, C.byref(prm), C.byref(g), C.byref(pa), C.byref(part), C.byref(nodes), s))
        assert not spoilt().any()
        keep = a["v"][0, bad].clone()
        a["v"][0, bad] = value
        capi.check(L.pmpm_musl_map(ctx.ptr, C.byref(prm), C.byref(g), C.byref(pa), C.byref(pb), C.byref(part),
                                   C.byref(nodes), s))
        bad_nodes = spoilt()
        assert bad_nodes.any() and not (bad_nodes & ~window).any(), (value, np.nonzero(bad_nodes & ~window)[0])
        a["v"][0, bad] = keep
