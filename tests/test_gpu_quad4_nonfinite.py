"""GPU test: in products of blocks up to 4x4 infinities and NaNs reach exactly the
results that use them.

One matrix step covers 16 block pairs, those with an absent block as zeros. Both
operands get infinities and NaNs; the results' non-finite elements and infinities must be the oracle's, and the finite ones within the
bars of the mode: 1e-12 (FP64, a few thousand terms of 1.1e-16), 2e-5 and 2e-6
(FP32 operands, FP32 and FP64 sums: 6e-8 per operand and term).
"""
import numpy as np
import pytest

import cqmm
import oracle
from cases import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags,bar", [(0, 1e-12), (cqmm.CQMM_FP32, 2e-5),
                                       (cqmm.CQMM_FP32 | cqmm.CQMM_FP32_ACC64, 2e-6)])
@pytest.mark.parametrize("natoms,ra,rb,rc", [(1, 4.0, 5.0, 3.0), (41, 6.0, 7.0, 9.0), (27, 13.0, 13.0, 13.0),
                                             (60, 5.0, 5.0, 10.0)])
@pytest.mark.parametrize("nsf", [4, 3, ((4, .6), (1, .4))])
@pytest.mark.parametrize("mt", [1, 2])
def test_nonfinite_values_stay_in_their_products(mt, nsf, natoms, ra, rb, rc, flags, bar):
    case = Case(natoms, nsf, ra, rb, rc, mt, seed=19)
    plan = cqmm.Plan(case.desc)
    sizes = set(case.nsf.tolist())
    assert plan.info().tile_family == (cqmm.TILES_DENSE4 if sizes == {4} else cqmm.TILES_DENSE_MIXED)
    a, b, c = case.values()
    left = a if mt == 1 else c
    left[min(50, len(left) - 1)] = np.inf
    left[len(left) // 2] = np.nan
    left[len(left) * 3 // 4] = -np.inf
    b[len(b) // 3] = np.inf
    x, y, z = a.copy(), b.copy(), c.copy()
    with np.errstate(invalid="ignore"):
        oracle.mat_mult(case.desc, x, y, z)
    ref = z if mt == 1 else x
    x, y, z = a.copy(), b.copy(), c.copy()
    out = z if mt == 1 else x
    out[:] = 7.0
    plan.mat_mult(x, y, z, flags)
    plan.close()
    np.testing.assert_array_equal(np.isnan(out), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(out), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(out), np.isneginf(ref))
    fine = np.isfinite(ref)
    print(f"type {mt}, {natoms} atoms: {np.count_nonzero(~fine)} of {ref.size} not finite", flush=True)
    if fine.any():
        top = np.abs(ref[fine]).max(initial=1e-300)
        assert np.abs(out[fine] - ref[fine]).max() <= bar * top
