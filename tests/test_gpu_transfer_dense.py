"""GPU parity of the larger 3D P2G tiles (8 x 2 x 4 cells, taken from 16,385
particles on) on grids smaller than a tile, ragged in every axis and two or
three nodes wide, with hundreds of particles in every cell, boundary cells
included (windows that leave the grid and wrap around through the linear index,
usl_inline.h:122-126). Bar: field-scaled relative error after 3 steps against
the FP32 oracle <= 1e-4, as the other multi-step runs."""
import numpy as np
import pytest

from tests import scenarios as S

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("sf", ["linear", "quadratic", "cubic"])
@pytest.mark.parametrize("musl", [False, True])
@pytest.mark.parametrize("cells", [(2, 3, 2), (3, 2, 5), (4, 2, 4), (9, 5, 5), (19, 3, 6)])
def test_dense_small_grids(oracle_mod, cells, musl, sf):
    rng = np.random.default_rng(sum(cells))
    h, n = 0.1, 16500
    span = np.array(cells) * h
    pos = rng.uniform(0.0, 1.0, size=(n, 3)) * (span - 0.004) + 0.002
    spec = S.Spec(dim=3, origin=[0.0] * 3, end=list((np.array(cells) - 0.75) * h), cell_size=h, shape_function=sf, dt=1e-4,
                  ppc=n // int(np.prod(cells)), positions=pos, velocities=rng.normal(0.0, 0.2, size=(n, 3)),
                  materials=[("LinearElastic", {"density": 1000.0, "E": 1e5, "pois": 0.3})],
                  bcs=[("Gravity", {"gravity": [0.0, 0.0, -9.81]})], musl=musl)
    print(f"\n[gpu-test] dense cells={cells} {sf} {'MUSL' if musl else 'USL'}", flush=True)
    pm, solver = S.build_product(spec)
    sim = S.build_oracle(oracle_mod, spec, "f32")
    solver.solve_nsteps(3)
    for _ in range(3):
        sim.step()
    got, ref = S.product_state(solver), S.oracle_state(sim)
    for k in S.FIELDS:
        assert S.max_rel_err(got[k], ref[k]) <= 1e-4, k
