"""How step_ssprk3 launches its steps: on the stream (1 or 2 steps, or up to 8
with a dt that has no graphs) or as graphs of 32 steps and of the remainder,
kept until dt, the limiter, its eps or the launch configuration changes.  One
solver goes through all of it; after every call its state equals, bit for
bit, that of a solver that launches the same stages one by one."""
import numpy as np
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph

from test_gpu_parity import random_state

pytestmark = pytest.mark.gpu

CASES = {
    "euler_2d_p3": (ph.Euler(flux_type=ph.FLUX_HLLEC), 3, (9, 7)),
    "glm_2d_p2": (ph.MHDGLM2D(c_h=1.3, alpha_d=1.3 / 0.18), 2, (6, 5)),
    "euler_3d_p2": (ph.Euler(flux_type=ph.FLUX_HLLE), 2, (3, 3, 2)),
}


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("name", list(CASES))
def test_every_route_steps_alike(name, precision):
    phys, P, n = CASES[name]
    L = (1.0, 0.8, 1.2)[:len(n)]
    dt = 0.02 * min(L) / max(n) / (2 * P + 1)
    with M.Solver(n, L, phys, P=P, precision=precision) as a, M.Solver(n, L, phys, P=P, precision=precision) as b:
        q = random_state(phys, a.num_elements, a.NP, np.random.default_rng(6), len(n))
        for s in (a, b):
            s.set_state(q.astype(np.float32).astype(np.float64))

        def both(what, f=None, steps=0, h=dt):
            print(name, precision, what, steps, flush=True)
            if f:
                f(a), f(b)
            if steps:
                a.step_ssprk3(h, steps)
                for _ in range(steps):
                    for st in range(3):
                        b.rk_stage(st, h)
            x = a.get_state()
            assert np.isfinite(x).all()
            assert np.array_equal(x, b.get_state()), what

        both("new dt, on the stream", steps=4)
        both("the same dt again, as a graph", steps=4)
        both("its graphs are there", steps=8)
        for k in range(2):
            both("alternating dt, on the stream", steps=3, h=0.9 * dt)
            both("the first dt, its graphs kept", steps=4)
        both("one step", steps=1)
        both("two", steps=2, h=0.8 * dt)
        both("beyond the first-use limit", steps=9, h=0.7 * dt)
        both("full graph and remainder", steps=37)
        both("the limiter on: graphs of before do not fit", lambda s: s.enable_cell_limiter(True, 0.1), 37)
        both("limited, a step", steps=1)
        both("another eps", lambda s: s.enable_cell_limiter(True, 0.01), 33)
        both("prepared, then stepped", lambda s: s.prepare_steps(0.6 * dt, 5), 5, 0.6 * dt)
        both("nothing to prepare for two", lambda s: s.prepare_steps(0.5 * dt, 2), 2, 0.5 * dt)
        both("another launch configuration", lambda s: setattr(s, "launch_config", 2), 33)
        both("the same on the stream", steps=2)
        both("the limiter off", lambda s: s.enable_cell_limiter(False), 33)
        both("a dt of its own each call", steps=5, h=0.55 * dt)
        both("off and on", lambda s: s.enable_cell_limiter(True, 0.1), 9)
        # the timing calls: as many steps of the same kind, limiter off
        both("bench loop", lambda s: s.enable_cell_limiter(False))
        a.bench_step_loop(dt, 2, 5)
        for _ in range(7):
            for st in range(3):
                b.rk_stage(st, dt)
        both("after the bench loop", steps=12)
        both("and limited", lambda s: s.enable_cell_limiter(True, 0.1), 12)
