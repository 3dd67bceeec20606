"""Uniform 4, 9, 13 and 16 blocks: one wavefront per 4x4 output blocks.

The sizes are those where the record lists, the ring of operand blocks and the
quadrants have their edges: one and two atoms (lists of a few records, most of a
quadrant absent), an atom count that is no multiple of 4 or 8, and ranges at
which every quadrant is full (records of eight blocks, lists of several hundred
words). Bars relative to the largest result: 1e-12 for FP64 (a few thousand
terms of 1.1e-16); 2e-5 and 2e-6 for FP32 operands with FP32 and FP64 sums
(6e-8 per operand and per 16-term product, times the terms of one sum); 5e-5 for
split BF16 (16 significant bits per operand).
"""
import numpy as np
import pytest

import cqmm
import oracle
from cases import Case

pytestmark = pytest.mark.gpu

MODES = ((0, 1e-12), (cqmm.CQMM_FP32, 2e-5), (cqmm.CQMM_FP32 | cqmm.CQMM_FP32_ACC64, 2e-6),
         (cqmm.CQMM_FP32 | cqmm.CQMM_BF16X3, 5e-5))


@pytest.mark.parametrize("natoms,ra,rb,rc", [(1, 4.0, 5.0, 3.0), (2, 3.0, 3.0, 3.0), (41, 6.0, 7.0, 9.0),
                                             (27, 13.0, 13.0, 13.0)])
@pytest.mark.parametrize("nsf", [4, 9, 13, 16])
@pytest.mark.parametrize("mt", [1, 2])
def test_wave_tiles(natoms, ra, rb, rc, nsf, mt):
    case = Case(natoms, nsf, ra, rb, rc, mt, seed=61)
    plan = cqmm.Plan(case.desc)
    info = plan.info()
    assert info.kernel == cqmm.KERNEL_TILE
    print(f"natoms={natoms} nsf={nsf} ranges={ra},{rb},{rc} type={mt}: {info.n_triplets} products, "
          f"{info.n_loads} blocks copied", flush=True)
    a, b, c = case.values()
    # One block of the left operand (type 1: A, type 2: C) with an infinity and
    # a NaN: they reach exactly the results that use them.
    left = a if mt == 1 else c
    # (4x4 blocks multiply them by the zeros of absent blocks too.)
    for bad in (False, True) if nsf != 4 else (False,):
        if bad:
            blk = left.reshape(-1, nsf * nsf)
            blk[min(3, len(blk) - 1), [1, -1]] = np.inf, np.nan
        x, y, z = a.copy(), b.copy(), c.copy()
        oracle.mat_mult(case.desc, x, y, z)
        ref = (z if mt == 1 else x).copy()
        top = np.abs(ref[np.isfinite(ref)]).max(initial=1e-300)
        for flags, bar in MODES[:1] if bad else MODES[:3] if nsf == 4 else MODES:
            x, y, z = a.copy(), b.copy(), c.copy()
            out = z if mt == 1 else x
            out[:] = 7.0
            plan.mat_mult(x, y, z, flags)
            fine = np.isfinite(ref)
            np.testing.assert_array_equal(np.isfinite(out), fine)
            err = np.abs(out[fine] - ref[fine]).max(initial=0.0) / top
            print(f"  flags {flags} bad {bad}: rel err {err:.3e}", flush=True)
            assert err <= bar
    plan.close()
