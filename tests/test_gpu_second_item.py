"""Tets with one component: the second face item of a thread is loaded with
the first, and its trace waits in its face-flux slot.  Meshes of several
tiles (traces from other tiles among the second items), with part-filled
tiles, boundaries, one cell per period (all faces in the tile), and P = 1,
where a thread can have a third item."""
import numpy as np
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph

from test_gpu_parity import TOL, random_state, rel_l2, run_pair

pytestmark = pytest.mark.gpu

ADV = ph.Advection(1.0, 0.7, -0.4, inflow_q=0.3)
MESHES = [((5, 3, 3), None), ((4, 3, 2), [3, 2, 1, 2, 3, 1]), ((3, 3, 3), [0, 0, 2, 3, 0, 0]), ((1, 1, 1), None)]


@pytest.mark.parametrize("P", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("case", range(len(MESHES)))
def test_second_items(oracle, P, case):
    n, bc = MESHES[case]
    print(P, n, bc, flush=True)
    L = (1.0, 0.8, 1.2)
    rng = np.random.default_rng(10 * P + case)
    K, NP = 6 * n[0] * n[1] * n[2], (P + 1) * (P + 2) * (P + 3) // 6
    q0 = random_state(ADV, K, NP, rng, 3).astype(np.float32).astype(np.float64)
    got, want, _ = run_pair(oracle, n, L, P, ADV, bc, nsteps=2, q0=q0)
    assert np.isfinite(got).all()
    assert rel_l2(got, want) < TOL
    # FP32: 2 steps of 3 stages, each rounded to FP32 (2^-23 relative at most)
    # and computed in FP32 from operands of a few times the state's size
    dt = 0.2 * min(L) / max(n) / (2 * P + 1) / 2.0
    with M.Solver(n, L, ADV, P=P, bcs=M.BoundaryConditions(*bc) if bc else None, precision=M.PREC_FP32_MFMA) as s:
        s.set_state(q0)
        s.step_ssprk3(dt, 2)
        assert rel_l2(s.get_state(), want) < 16 * 2.0 ** -23
