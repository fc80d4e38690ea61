"""Limited steps on meshes of several ragged tiles, where the stage kernel
computes the factors of its own elements and of those behind its tile's
faces: against the oracle (1e-12 over three steps, the bar of the limited
parity tests), against the per-stage API, which stores the limited state
after every stage, and against the batch engine, both bit for bit."""
import numpy as np
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph
from mojoxm_amd.batch import Batch

from test_gpu_parity import random_state, rel_l2

pytestmark = pytest.mark.gpu

EULER = ph.Euler(flux_type=ph.FLUX_HLLE)
CASES = {
    "euler_2d_p1": (EULER, 1, (23, 9), (2, 2, 1, 1)),
    "euler_2d_p3": (EULER, 3, (17, 13), None),
    "sw_2d_p2": (ph.ShallowWater2D(hll=True), 2, (19, 11), (1, 1, 1, 1)),
    "maxwell_2d_p4": (ph.Maxwell2D(), 4, (9, 7), (1, 1, 0, 0)),
    "euler_3d_p1": (EULER, 1, (7, 3, 5), None),
    "euler_3d_p2": (EULER, 2, (4, 3, 3), (2, 2, 1, 1, 0, 0)),
    "mhd_3d_p3": (ph.IdealMHD(c_h=1.7), 3, (3, 2, 3), None),
}


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("name", list(CASES))
def test_limited_tiles(oracle, name, precision):
    phys, P, n, bc = CASES[name]
    print(f"{name} {precision}", flush=True)
    nd, L = len(n), (1.0, 0.8, 1.2)[:len(n)]
    bcs = (M.BoundaryConditions if nd == 3 else M.BoundaryConditions2D)(*bc) if bc else None
    dt = 0.05 * min(L) / max(n) / (2 * P + 1)
    with M.Solver(n, L, phys, P=P, bcs=bcs, precision=precision) as s:
        q = random_state(phys, s.num_elements, s.NP, np.random.default_rng(5), nd)
        q = q.astype(np.float32).astype(np.float64)
        s.enable_cell_limiter(True, 0.1)
        s.set_state(q)
        s.step_ssprk3(dt, 3)
        got = s.get_state()
        s.set_state(q)
        for _ in range(3):
            for st in range(3):
                s.rk_stage(st, dt)
        assert np.array_equal(s.get_state(), got)
    with Batch(precision) as b:
        ids = [b.add(n, L, phys, P, q, dt, k, bcs=bcs, limiter=True, eps=0.1) for k in (3, 5)]
        b.step(1)
        b.get_state(ids[0])  # stores the limited state in between
        b.step(2)
        for i in ids:
            assert np.array_equal(b.get_state(i), got)
    if precision == M.PREC_FP64:
        om = oracle.Mesh(nd, P, n, L, list(bc) if bc else None)
        want = om.step(phys.phys_id, phys.params(), q, dt, 3, limiter=True)
        assert rel_l2(got, want) < 1e-12
