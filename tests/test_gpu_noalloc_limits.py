"""GPU: pmpm_step_noalloc on grids of a single row, near the end of its
workspace, where the P2G tiles' partials do not fit it and every particle is
deposited over its own window instead; and with particles left of the origin,
whose sums go to the step's node arrays. Bar: positions, velocities, stresses
and F within a field-scaled relative error of 1e-5 of pmpm_step with a context
(the same sums in another order), two steps in a row, USL and MUSL."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _run(dim, sf, cells, n, musl, noalloc):
    from pyroclastmpm_amd import capi
    dev = torch.device("cuda")
    rng = np.random.default_rng(3)
    g = capi.Grid()
    g.cell_size = g.inv_cell_size = 1.0
    for a in range(3):
        g.num_cells[a] = cells[a] if a < dim else 1
    nn = g.num_cells_total = int(np.prod(cells))
    # clusters of a few cells: at both ends of the slowest axis, and left of the origin
    pos = rng.uniform(0.1, 0.9, (n, dim)) * np.array([min(c, 6) for c in cells[:dim]])
    pos[n // 2:, 0] += max(0, cells[0] - 8)
    pos[:20, 0] = -rng.uniform(0.05, 0.9, 20)
    f = lambda *s: torch.zeros(*s, device=dev)
    i32 = lambda m: torch.zeros(m, dtype=torch.int32, device=dev)
    put = lambda v: torch.from_numpy(np.ascontiguousarray(v, dtype=np.float32)).to(dev)

    def particles(fill):
        t = {"x": f(dim, n), "v": f(dim, n), "stress": f(6, n), "F": f(dim * dim, n), "L": f(dim * dim, n), "mass": f(n) + 1,
             "volume": f(n) + 0.1, "volume0": f(n) + 0.1, "color": torch.zeros(n, dtype=torch.uint8, device=dev),
             "flags": torch.full((n,), capi.PF_ACTIVE, dtype=torch.uint8, device=dev),
             "id": torch.arange(n, dtype=torch.int32, device=dev)}
        if fill:
            t["x"].copy_(put(pos.T))
            t["v"].copy_(put(rng.normal(0, 0.1, (dim, n))))
            t["stress"].copy_(put(rng.normal(0, 0.1, (6, n))))
            for a in range(dim):
                t["F"][a * dim + a] = 1.0
        return t, capi.Particles(n, *[t[k].data_ptr() for k in ["x", "v", "stress", "F", "L", "mass", "volume", "volume0",
                                                                "color", "flags", "id"]])

    sets = [particles(True), particles(False)]
    sp = {"hash": i32(n), "hash_sorted": i32(n), "sorted": i32(n), "cell_start": i32(nn), "cell_end": i32(nn)}
    part = capi.Spatial(*[sp[k].data_ptr() for k in sp], None)
    nd = {"mass": f(nn) + 5, "mom": f(dim * nn) + 5, "mom_nt": f(dim * nn) + 5, "vel": f(capi.node_vel_stride(dim) * nn)}
    nodes = capi.Nodes(*[nd[k].data_ptr() for k in nd])
    prm = capi.Params()
    prm.dim, prm.shape_fn, prm.dt, prm.alpha = dim, capi.SF[sf], 1e-3, 0.99
    prm.small_mass_cutoff, prm.node_types_built, prm.wrap_quirk = 1e-9, int(sf == "cubic"), 1
    prm.num_materials = 1
    prm.materials[0].kind = capi.MAT_LINEAR_ELASTIC
    for k, v in enumerate((100.0, 50.0, 130.0)):
        prm.materials[0].p[k] = v
    prm.num_bcs = 1
    prm.bcs[0].kind = capi.BC_GRAVITY
    prm.bcs[0].f[dim - 1] = -9.81
    s, L = torch.cuda.current_stream().cuda_stream, capi.lib()
    ctx = None if noalloc else capi.Context(n, nn)
    for k in range(2):
        a, b = sets[k][1], sets[1 - k][1]
        args = (C.byref(prm), C.byref(g), int(musl), C.byref(a), C.byref(b), C.byref(part), C.byref(nodes), s)
        capi.check(L.pmpm_step_noalloc(*args) if noalloc else L.pmpm_step(ctx.ptr, *args), "step")
    torch.cuda.synchronize()
    t = sets[0][0]
    back = torch.argsort(t["id"].long())
    return {k: t[k][:, back].double().cpu().numpy() for k in ("x", "v", "stress", "F")}


@pytest.mark.parametrize("musl", [False, True])
@pytest.mark.parametrize("dim, sf, cells", [(2, "linear", (1500000, 1)), (2, "cubic", (700000, 1)), (2, "quadratic", (60, 40)),
                                            (3, "quadratic", (520, 1, 520)), (3, "linear", (25, 1, 28000)),
                                            (3, "cubic", (30, 20, 10))])
def test_noalloc_near_its_limit(dim, sf, cells, musl):
    print(f"\n[gpu-test] noalloc {dim}D {sf} {cells} {'MUSL' if musl else 'USL'}", flush=True)
    want, got = (_run(dim, sf, cells, 3000, musl, na) for na in (False, True))
    for k in want:
        assert np.isfinite(want[k]).all() and np.abs(want[k]).max() > 0
        e = np.abs(got[k] - want[k]).max() / np.abs(want[k]).max()
        assert e <= 1e-5, (k, e)
