"""The 3D limiter, whose factor is the minimum over all components: every order
and every number of components, on meshes of several ragged tiles with
boundaries (neighbours that are the element itself) and without, against the
oracle in both forms (the bars of the limited parity tests: 1e-12, FP32
1e-5), and the per-stage calls and a batch against it bit for bit."""
import numpy as np
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph
from mojoxm_amd.batch import Batch

from test_gpu_fp32 import TOL32
from test_gpu_parity import TOL, random_state, rel_l2

pytestmark = pytest.mark.gpu

PHYS = {
    "advection": ph.Advection(1.0, 0.7, -0.4, inflow_q=0.3),
    "sw": ph.ShallowWater(),
    "euler": ph.Euler(flux_type=ph.FLUX_HLLE),
    "maxwell": ph.Maxwell(),
    "mhd": ph.IdealMHD(c_h=1.7),
    "two_fluid": ph.FiveMomentTwoFluid(c_light=2.0, c_h=1.5, alpha_d=0.5),
}
MESHES = [((3, 2, 3), None), ((2, 3, 2), (2, 2, 1, 1, 0, 0)), ((1, 1, 1), None)]


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("P", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("name", list(PHYS))
def test_limited_components(oracle, name, P, precision):
    phys, L = PHYS[name], (1.0, 0.8, 1.2)
    for n, bc in MESHES:
        print(name, P, n, bc, precision, flush=True)
        bcs = M.BoundaryConditions(*bc) if bc else None
        dt = 0.05 * min(L) / max(n) / (2 * P + 1)
        with M.Solver(n, L, phys, P=P, bcs=bcs, precision=precision) as s:
            q = random_state(phys, s.num_elements, s.NP, np.random.default_rng(P), 3)
            q = q.astype(np.float32).astype(np.float64)
            s.enable_cell_limiter(True, 0.1)
            s.set_state(q)
            s.step_ssprk3(dt, 2)
            got = s.get_state()
            s.set_state(q)
            for _ in range(2):
                for st in range(3):
                    s.rk_stage(st, dt)
            assert np.array_equal(s.get_state(), got)
        with Batch(precision) as b:
            i = b.add(n, L, phys, P, q, dt, 2, bcs=bcs, limiter=True, eps=0.1)
            b.step(2)
            assert np.array_equal(b.get_state(i), got)
        om = oracle.Mesh(3, P, n, L, list(bc) if bc else None)
        want = om.step(phys.phys_id, phys.params(), q, dt, 2, limiter=True, eps=0.1)
        assert rel_l2(got, want) < (TOL if precision == M.PREC_FP64 else TOL32)


PHYS_2D = {
    "euler": ph.Euler(flux_type=ph.FLUX_HLLE),
    "sw": ph.ShallowWater2D(hll=True),
    "maxwell": ph.Maxwell2D(),
    "glm": ph.MHDGLM2D(c_h=1.3, alpha_d=1.3 / 0.18),
}
MESHES_2D = [((17, 9), None), ((13, 11), (2, 2, 1, 1)), ((1, 1), None)]


@pytest.mark.parametrize("P", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("name", list(PHYS_2D))
def test_limited_triangles_fp32(oracle, name, P):
    """The FP32 form on triangles (one limited component) against the oracle:
    ragged tiles, boundaries, every order."""
    phys, L = PHYS_2D[name], (1.0, 0.8)
    for n, bc in MESHES_2D:
        print(name, P, n, bc, flush=True)
        bcs = M.BoundaryConditions2D(*bc) if bc else None
        dt = 0.05 * min(L) / max(n) / (2 * P + 1)
        with M.Solver(n, L, phys, P=P, bcs=bcs, precision=M.PREC_FP32_MFMA) as s:
            q = random_state(phys, s.num_elements, s.NP, np.random.default_rng(P), 2)
            q = q.astype(np.float32).astype(np.float64)
            s.enable_cell_limiter(True, 0.1)
            s.set_state(q)
            s.step_ssprk3(dt, 2)
            got = s.get_state()
        om = oracle.Mesh(2, P, n, L, list(bc) if bc else None)
        want = om.step(phys.phys_id, phys.params(), q, dt, 2, limiter=True, eps=0.1)
        assert rel_l2(got, want) < TOL32
