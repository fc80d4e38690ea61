"""Tiles of meshes that are no multiple of the tile's block of cells: what
whole blocks leave over is cut into tiles of other shapes.  Building the
tables of a mesh checks that every element lies in one tile and that every
face slot of a tile is written once, and needs no GPU."""
import itertools

import numpy as np
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph
from mojoxm_amd.batch import Batch, footprint

from test_gpu_parity import TOL, random_state, rel_l2, run_pair

EULER = ph.Euler(flux_type=ph.FLUX_HLLEC, inflow=(1.0, 0.1, 0.2, 0.0, 2.5))


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("P", [1, 2, 3, 4, 5])
def test_every_mesh_is_covered(P, precision):
    for n in itertools.product([1, 2, 5, 6, 7, 13], [1, 3, 4, 11]):
        for bc in (None, M.BoundaryConditions2D(1, 2, 3, 1)):
            assert footprint(n, (1.0, 1.0), EULER, P, precision, bcs=bc) > 0
    for n in itertools.product([1, 2, 3, 5], [1, 2, 3], [1, 2, 5]):
        for bc in (None, M.BoundaryConditions(1, 2, 3, 1, 0, 0)):
            assert footprint(n, (1.0, 1.0, 1.0), EULER, P, precision, bcs=bc) > 0


@pytest.mark.parametrize("n", [(17, 17), (19, 19), (31, 33), (67, 29), (19, 19, 19), (7, 5, 9)])
def test_ragged_meshes_take_few_tiles(n):
    # per-tile memory of whole blocks: 4 x 3 squares, 2 x 1 x 1 cubes
    whole = (48, 48) if len(n) == 2 else (8, 8, 8)
    per = [footprint(k, (1.0,) * len(n), EULER, 3, M.PREC_FP32_MFMA) / np.prod(k) for k in (whole, n)]
    # 12 cells a tile: at worst 26 tiles where 24.1 would hold 17 x 17
    # squares; 2 cells a tile: one tile more than half the cells at most per
    # plane left over.  The per-instance tables are below 1 % of either.
    assert per[1] < 1.10 * per[0]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("P,n", [(1, (39, 41)), (2, (25, 19)), (3, (17, 17)), (3, (13, 29)), (4, (15, 17)), (5, (11, 13)),
                                 (2, (5, 5, 3)), (3, (3, 5, 3)), (4, (3, 3, 5))])
def test_ragged_meshes_give_the_same_bits(P, n, precision):
    # alone, a small mesh keeps blocks cut off at its edge; in a batch its
    # remainders are tiles of other shapes
    L = (1.0, 0.8, 1.2)[:len(n)]
    dt = 0.1 * min(L) / max(n) / (2 * P + 1)
    B = M.BoundaryConditions if len(n) == 3 else M.BoundaryConditions2D
    for bcs in (None, B(*[1, 2, 3, 1, 2, 2][:2 * len(n)])):
        print(P, n, precision, bcs, flush=True)
        with M.Solver(n, L, EULER, P=P, bcs=bcs, precision=precision) as s:
            q = random_state(EULER, s.num_elements, s.NP, np.random.default_rng(P), len(n))
            q = q.astype(np.float32).astype(np.float64)
            s.set_state(q)
            s.step_ssprk3(dt, 2)
            want = s.get_state()
        with Batch(precision) as b:
            i = b.add(n, L, EULER, P, q, dt, 2, bcs=bcs)
            b.step(2)
            assert np.isfinite(want).all()
            assert np.array_equal(b.get_state(i), want)


@pytest.mark.gpu
@pytest.mark.parametrize("P,n", [(3, (61, 59)), (2, (9, 11, 13))])
def test_large_ragged_mesh_matches_the_oracle(oracle, P, n):
    # more blocks than CUs: the remainders of a mesh alone are cut as well
    print(P, n, flush=True)
    got, want, _ = run_pair(oracle, n, (1.0, 0.8, 1.2)[:len(n)], P, EULER, None, nsteps=1, seed=P)
    assert np.isfinite(got).all()
    assert rel_l2(got, want) < TOL


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_FP32_MFMA])
@pytest.mark.parametrize("L", [(1e155, 1e155, 1e-10), (1e160, 1e-100, 1e-100), (1e-100, 1e-100, 1e-100),
                               (1e-155, 1e-155), (1e160, 1e160), (1.0 / 3.0, 7.3e-3), (0.7, 1e6, 3.1e-5)])
def test_extreme_extents_are_accepted(L, precision):
    """The geometry of a mesh is found again by its bits: extents whose face
    normals overflow to NaN make tables as any others do."""
    n = (3, 2, 5)[:len(L)]
    for bc in (None, (M.BoundaryConditions(1, 2, 3, 1, 1, 2) if len(L) == 3 else M.BoundaryConditions2D(1, 2, 3, 1))):
        assert footprint(n, L, EULER, 2, precision, bcs=bc) > 0
