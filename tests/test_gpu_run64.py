"""GPU test: CQMM_FP32_RUN64 adds every product in FP64, as CQMM_FP32_ACC64 does.

The two flags give the same bits on every schedule, and the bar is that of FP64
sums of FP32 products, 2e-6 of the largest result (6e-8 per operand and term).
"""
import numpy as np
import pytest

import cqmm
import oracle
from cases import Case

pytestmark = pytest.mark.gpu

MIX = ((4, .5), (9, .25), (13, .25))


@pytest.mark.parametrize("nsf", [4, 9, 13, 16, 22, MIX])
@pytest.mark.parametrize("mt", [1, 2])
def test_run64_is_acc64(nsf, mt):
    case = Case(41, nsf, 6.0, 7.0, 9.0, mt, seed=61)
    plan = cqmm.Plan(case.desc)
    a, b, c = case.values()
    outs = []
    for flags in (cqmm.CQMM_FP32 | cqmm.CQMM_FP32_ACC64, cqmm.CQMM_FP32 | cqmm.CQMM_FP32_RUN64):
        x, y, z = a.copy(), b.copy(), c.copy()
        plan.mat_mult(x, y, z, flags)
        outs.append(z if mt == 1 else x)
    plan.close()
    np.testing.assert_array_equal(outs[0], outs[1])
    x, y, z = a.copy(), b.copy(), c.copy()
    oracle.mat_mult(case.desc, x, y, z)
    ref = z if mt == 1 else x
    assert np.abs(outs[1] - ref).max() <= 2e-6 * np.abs(ref).max()
