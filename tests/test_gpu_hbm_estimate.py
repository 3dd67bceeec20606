"""GPU test: a solve's measured device peak stays within its admission estimate.

One case per schedule family (below 4x4, 4x4, mixed-size kernel, wavefront
kernel) at ranges where its products have the most bytes each: short ranges for
the small blocks, a long density matrix for the others.
"""
import pytest

from cqmm import serve as sv

pytestmark = pytest.mark.gpu

SHORT = dict(r_S=4.5, r_H=4.5, r_L=6.0)
LONG = dict(r_S=6.0, r_H=6.0, r_L=16.0)


@pytest.mark.parametrize("natoms,nsf,ranges", [(2000, 1, SHORT), (500, 2, SHORT), (24, 3, LONG), (48, 4, LONG),
                                               (48, 5, LONG), (300, 13, SHORT)])
def test_peak_within_the_estimate(natoms, nsf, ranges):
    params = sv.default_params(precision=1, max_iter=1, **ranges)
    r = sv.purify(natoms, nsf, 5, params)
    print(f"{natoms} atoms x {nsf}: peak {r['hbm_peak']} estimate {r['hbm_estimate']}", flush=True)
    assert r["status"] == 0
    assert 0 < r["hbm_peak"] <= r["hbm_estimate"]
