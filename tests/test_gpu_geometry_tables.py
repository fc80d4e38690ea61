"""The stage kernel's per-lattice geometry (one table per instance, an
element's entry found from its place in its lattice cell): meshes of
different spacing and boundaries in one batch arena give the bits each gives
alone, also where a tile holds less than a cell, so that tiles and arena
ranges start anywhere in a cell (3D, P = 5: 4 of 6 tets; two-fluid, P = 4: 4)."""
import numpy as np
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph
from mojoxm_amd.batch import Batch

from test_gpu_parity import random_state

pytestmark = pytest.mark.gpu

EULER = ph.Euler(flux_type=ph.FLUX_HLLEC, inflow=(1.0, 0.1, 0.2, 0.0, 2.5))
FLUID = ph.FiveMomentTwoFluid(c_light=2.0, c_h=1.5, alpha_d=0.5)
CASES = {
    "euler_p5": (EULER, 5, [((1, 1, 1), (1.0, 2.0, 3.0), None), ((2, 1, 3), (1.0, 0.7, 1.3), (2, 3, 1, 1, 0, 0)),
                            ((1, 2, 1), (0.5, 0.5, 0.5), (1, 1, 1, 1, 1, 1))]),
    "twofluid_p4": (FLUID, 4, [((1, 1, 1), (1.0, 2.0, 3.0), None), ((1, 2, 2), (1.0, 0.7, 1.3), (1, 1, 0, 0, 2, 2))]),
    "euler_2d_p3": (EULER, 3, [((3, 5), (1.0, 2.0), None), ((5, 2), (0.3, 0.4), (2, 3, 1, 1)), ((1, 1), (1.0, 1.0), None)]),
}


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("name", list(CASES))
def test_mixed_geometry_batch_matches_alone(name, precision):
    phys, P, meshes = CASES[name]
    rng = np.random.default_rng(17)
    want, items = [], []
    for n, L, bc in meshes:
        print(f"{name} {n} {bc} {precision}", flush=True)
        nd = len(n)
        bcs = (M.BoundaryConditions if nd == 3 else M.BoundaryConditions2D)(*bc) if bc else None
        dt = 0.02 * min(L) / max(n) / (2 * P + 1)
        with M.Solver(n, L, phys, P=P, bcs=bcs, precision=precision) as s:
            q = random_state(phys, s.num_elements, s.NP, rng, nd).astype(np.float32).astype(np.float64)
            s.set_state(q)
            s.step_ssprk3(dt, 3)
            want.append(s.get_state())
        items.append((n, L, bcs, q, dt))
    with Batch(precision) as b:
        ids = [b.add(n, L, phys, P, q, dt, 3, bcs=bcs) for n, L, bcs, q, dt in items]
        b.step(3)
        for i, w in zip(ids, want):
            assert np.array_equal(b.get_state(i), w)
