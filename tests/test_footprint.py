"""Device bytes of a batch instance (admission by memory budget).  The bounds
are what the instances took when the stage kernel read a geometry record per
face and per slot and the limiter kept one buffer's extrema: what fitted a
budget then still fits.  (3D limited FP64 instances of 6 components and more
keep 3 buffers' extrema and are up to 2 %, MHD 7 %, two-fluid 14 % larger than
then; the last rows bound those.)"""
import pytest

import mojoxm_amd as M
from mojoxm_amd import physics as ph
from mojoxm_amd.batch import footprint

F64, F32 = M.PREC_FP64, M.PREC_FP32_MFMA
ADV, EUL, SW, MX, MHD, TF = (ph.Advection(1.0, 0.7, -0.4), ph.Euler(), ph.ShallowWater(), ph.Maxwell(), ph.IdealMHD(),
                             ph.FiveMomentTwoFluid())
WALLS3, WALLS2 = M.BoundaryConditions(1, 2, 2, 1, 1, 1), M.BoundaryConditions2D(1, 2, 2, 1)
BOUNDS = [
    (EUL, 2, (1, 1), F64, True, WALLS2, 39710),
    (EUL, 3, (16, 16), F64, True, None, 871584),
    (EUL, 3, (37, 29), F32, False, WALLS2, 1806688),
    (EUL, 5, (3, 2), F32, True, None, 19040),
    (ADV, 2, (3, 2, 5), F32, False, None, 88208),
    (ADV, 1, (8, 8, 8), F32, True, None, 1214240),
    (SW, 1, (1, 1, 1), F32, True, WALLS3, 24308),
    (EUL, 1, (1, 1, 1), F32, False, None, 21104),
    (EUL, 1, (8, 8, 8), F32, True, WALLS3, 2565920),
    (EUL, 3, (3, 2, 5), F32, False, WALLS3, 357728),
    (EUL, 2, (13, 11, 7), F64, True, None, 11856720),
    (EUL, 1, (8, 8, 8), F64, True, WALLS3, 3487520),
    (EUL, 5, (3, 2, 5), F64, True, WALLS3, 1324548),
    (MX, 2, (8, 8, 8), F32, True, WALLS3, 3810592),
    (MHD, 1, (8, 8, 8), F32, True, None, 3217184),
    (TF, 1, (8, 8, 8), F32, True, None, 5408032),
    (TF, 2, (13, 11, 7), F32, True, WALLS3, 19473280),
    (TF, 1, (3, 2, 5), F64, False, None, 447488),
    (MX, 1, (8, 8, 8), F64, True, None, 4072512),
    (MHD, 1, (8, 8, 8), F64, True, None, 4828224),
    (MHD, 3, (8, 8, 8), F64, True, None, 15583552),
    (TF, 1, (8, 8, 8), F64, True, None, 8964928),
    (TF, 3, (8, 8, 8), F64, True, None, 29166912),
]


@pytest.mark.parametrize("phys,P,n,precision,limiter,bcs,most", BOUNDS)
def test_instances_fit_their_former_budget(phys, P, n, precision, limiter, bcs, most):
    assert footprint(n, (1.0,) * len(n), phys, P, precision, limiter=limiter, bcs=bcs) <= most
