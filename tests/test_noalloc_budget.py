"""CPU: which steps pmpm_step_noalloc accepts. A step is charged by its particle
count and grid against PMPM_NOALLOC_SCRATCH_BYTES before anything is launched;
the rule is part of the entry's contract (what a caller may ask for does not
move with the kernels' tilings), so it is restated here and held at its edge:
the largest accepted and the smallest refused grid of several shapes. Without a
GPU an accepted step ends at the first HIP call (PMPM_ERR_HIP)."""
import ctypes as C

import pytest

from pyroclastmpm_amd import capi

torch = pytest.importorskip("torch")

LIMIT = capi.NOALLOC_SCRATCH_BYTES
div = lambda a, b: -(-a // b)


def _charge(dim, sf, typed, c, n):
    """Bytes, in pieces of whole 256 bytes."""
    nodes, span = c[0] * c[1] * c[2], 2 if sf == "linear" else 4
    tiles = []

    def tile(tx):
        t = div(c[0], tx) * (c[1] if dim > 1 else 1) * (div(c[2], 4) if dim > 2 else 1)
        tiles.append((t * (1 + 2 * dim) * (tx + span - 1) * (span if dim > 1 else 1) * (3 + span if dim > 2 else 1), t))

    tile({1: 256, 2: 256 // span, 3: 64 // span}[dim])
    if dim == 3 and typed:
        tile(8)
    wrap = 0 if dim < 2 else 3 * c[1] * c[2] + (3 * (c[0] - 3) * c[2] if dim > 2 and c[0] > 3 else 0)
    records = [8 * 64 * wrap, div(nodes, 4), 32 * (1 + wrap)] if typed and wrap else []
    words = [n, n, 1024 * div(n, 4096) + 1024, 4, max(t[0] for t in tiles), max(t[1] for t in tiles), *records, div(nodes, 4)]
    return sum(div(4 * w, 256) * 256 for w in words)


def _call(dim, sf, typed, c, n):
    prm, g = capi.Params(), capi.Grid()
    prm.dim, prm.shape_fn, prm.dt, prm.alpha = dim, capi.SF[sf], 1e-4, 0.99
    prm.node_types_built, prm.wrap_quirk = int(typed), 1
    g.cell_size = g.inv_cell_size = 1.0
    for a in range(3):
        g.num_cells[a] = c[a]
    g.num_cells_total = c[0] * c[1] * c[2]
    some = [256] * 14  # never read: the step ends before its first launch
    a, b = capi.Particles(n, *some), capi.Particles(n, *[512] * 14)
    sp, nd = capi.Spatial(*[256] * 6), capi.Nodes(*[256] * 5)
    return capi.lib().pmpm_step_noalloc(C.byref(prm), C.byref(g), 1, C.byref(a), C.byref(b), C.byref(sp), C.byref(nd), None)


@pytest.mark.skipif(torch.cuda.is_available(), reason="the arrays are no memory: only where no kernel can be launched")
@pytest.mark.parametrize("dim, sf, typed, shape, n", [
    (1, "linear", False, lambda k: (k, 1, 1), 1000), (2, "cubic", True, lambda k: (k, k + 7, 1), 50000),
    (2, "linear", False, lambda k: (k, 1, 1), 777), (2, "quadratic", False, lambda k: (k, 2, 1), 9),
    (3, "cubic", True, lambda k: (k, k // 2 + 1, k // 2 + 1), 16704), (3, "quadratic", False, lambda k: (k, 1, k), 40000),
    (3, "linear", False, lambda k: (25, 1, k), 148), (3, "linear", False, lambda k: (2 * k, k, k), 2000000)])
def test_accepted_steps(dim, sf, typed, shape, n):
    lo, hi = 1, 1 << 24
    assert _charge(dim, sf, typed, shape(lo), n) <= LIMIT
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if _charge(dim, sf, typed, shape(mid), n) <= LIMIT else (lo, mid)
    near = [k for k in range(max(1, lo - 2), hi + 3)] + [max(1, lo // 2), 2 * hi]
    for k in near:
        fits = _charge(dim, sf, typed, shape(k), n) <= LIMIT
        rc = _call(dim, sf, typed, shape(k), n)
        assert rc == (capi.PMPM_ERR_HIP if fits else capi.PMPM_ERR_WORKSPACE), (shape(k), fits)
        if not fits:
            assert b"PMPM_NOALLOC_SCRATCH_BYTES" in capi.lib().pmpm_last_error()
            assert str(_charge(dim, sf, typed, shape(k), n)).encode() in capi.lib().pmpm_last_error()
