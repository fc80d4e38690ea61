"""The limiter with stages called out of order: rk_stage accepts any stage
index, and each call limits what it stored, so no later call may limit a
buffer a second time.  set_state leaves nothing pending; handing a solver the
state it already has must change nothing."""
import numpy as np
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph

from test_gpu_parity import random_state

pytestmark = pytest.mark.gpu

CASES = {
    "euler_2d_p3": (ph.Euler(flux_type=ph.FLUX_HLLE), 3, (13, 9)),
    "sw_2d_p2": (ph.ShallowWater2D(hll=True), 2, (9, 7)),
    "euler_3d_p2": (ph.Euler(flux_type=ph.FLUX_HLLEC), 2, (4, 3, 3)),
    "mhd_3d_p1": (ph.IdealMHD(c_h=1.7), 1, (5, 3, 4)),
}


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("stages", [(2,), (1,), (2, 2), (1, 2), (0, 2, 1)])
def test_stages_out_of_order_limit_once(name, precision, stages):
    phys, P, n = CASES[name]
    print(name, precision, stages, flush=True)
    L = (1.0, 0.8, 1.2)[:len(n)]
    dt = 0.05 * min(L) / max(n) / (2 * P + 1)
    out = []
    for reload in (False, True):
        with M.Solver(n, L, phys, P=P, precision=precision) as s:
            q = random_state(phys, s.num_elements, s.NP, np.random.default_rng(3), len(n))
            s.set_state(q.astype(np.float32).astype(np.float64))
            s.enable_cell_limiter(True, 0.1)
            for st in (0, 1, 2) + stages:
                s.rk_stage(st, dt)
                if reload:
                    s.set_state(s.get_state())
            # the stage buffers show in what a last stage makes of them
            s.rk_stage(2, dt)
            out.append(s.get_state())
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("nsteps", [2, 9])
def test_a_stage_after_steps(name, precision, nsteps):
    """After a call of nsteps (on the stream, and as a graph) a single stage
    continues as it does after the same stages one by one."""
    phys, P, n = CASES[name]
    print(name, precision, nsteps, flush=True)
    L = (1.0, 0.8, 1.2)[:len(n)]
    dt = 0.05 * min(L) / max(n) / (2 * P + 1)
    for last in (1, 2):
        out = []
        for whole in (True, False):
            with M.Solver(n, L, phys, P=P, precision=precision) as s:
                q = random_state(phys, s.num_elements, s.NP, np.random.default_rng(4), len(n))
                s.set_state(q.astype(np.float32).astype(np.float64))
                s.enable_cell_limiter(True, 0.1)
                if whole:
                    s.step_ssprk3(dt, nsteps)
                else:
                    for _ in range(nsteps):
                        for st in range(3):
                            s.rk_stage(st, dt)
                s.rk_stage(last, dt)
                s.rk_stage(2, dt)
                out.append(s.get_state())
        assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("name", list(CASES))
def test_switching_leaves_nothing_pending(name, precision):
    """Off and on again, with a new state or steps in between, gives what a
    solver gives that is handed the same state with the limiter on."""
    phys, P, n = CASES[name]
    print(name, precision, flush=True)
    L = (1.0, 0.8, 1.2)[:len(n)]
    dt = 0.05 * min(L) / max(n) / (2 * P + 1)
    for between in ("nothing", "state", "steps", "timing"):
        out = []
        for switch in (True, False):
            with M.Solver(n, L, phys, P=P, precision=precision) as s:
                q, q2 = (random_state(phys, s.num_elements, s.NP, np.random.default_rng(k), len(n))
                         .astype(np.float32).astype(np.float64) for k in (5, 6))
                s.set_state(q)
                s.enable_cell_limiter(True, 0.1)
                s.step_ssprk3(dt, 3)
                if between == "state":
                    if switch:
                        s.enable_cell_limiter(False)
                    s.set_state(q2)
                elif between == "steps":
                    s.enable_cell_limiter(False)
                    s.step_ssprk3(dt, 2)
                    if not switch:  # nothing can be pending on a state that is set
                        s.enable_cell_limiter(True, 0.1)
                        s.set_state(s.get_state())
                elif between == "timing":
                    s.time_stage_kernel(dt, 1) if switch else None
                    s.set_state(q2)
                elif switch:
                    s.enable_cell_limiter(False)
                s.enable_cell_limiter(True, 0.1)
                s.step_ssprk3(dt, 2)
                s.rk_stage(2, dt)
                out.append(s.get_state())
        assert np.isfinite(out[0]).all()
        assert np.array_equal(out[0], out[1]), between
