"""Parent-grouped matrix-core M2L at the edges of its launch rule: scalar FP64
levels below and above 1024 blocks (directions split over the waves of a block,
or one tile per wave), column counts that leave part of a tile, source children
missing from whole tiles (surfaces), all translation shapes and dof counts of
the forward transform.  Plain form against the oracle at the FP64 parity bar,
mixed form against the plain one at its own bar.
"""
import pytest

import kifmm3d as K
from problems import densities, relerr, sphere, uniform_cube
from test_gpu_parity import PARITY, make_fmm, make_oracle

pytestmark = pytest.mark.gpu

MIXED_VS_PLAIN = 1e-6


@pytest.mark.parametrize("kt,np_,n,ptsmax,nrhs", [(111, 4, 1500, 40, 1), (111, 6, 9000, 40, 3), (111, 4, 30000, 40, 5),
                                                  (321, 4, 5000, 30, 3), (321, 8, 2000, 60, 1), (521, 6, 4000, 40, 1),
                                                  (521, 8, 2500, 60, 2)])
def test_grouped_form(kt, np_, n, ptsmax, nrhs):
    print(f"\n[case] kt={kt} np={np_} n={n} nrhs={nrhs}", flush=True)
    p, nor = (uniform_cube(n, 41), None) if kt == 111 else sphere(n, 42)
    ctr, rl = ((0.5, 0.5, 0.5), 1) if kt == 111 else ((0.0, 0.0, 0.0), 0)
    f = make_fmm(kt, np_, ptsmax, 10, ctr, rl, p, nor, p)
    for mode in (K.MODE_PLAIN, K.MODE_MIXED):
        f.set_settings(mode, -1, [1] * len(f.settings(mode)["m2l"]))
    den = densities(n, f.knl.sdof(), nrhs, 43)
    val = f.eval(den, nrhs=nrhs).reshape(nrhs, -1).copy()
    o = make_oracle(f, kt, np_, ptsmax, 10, ctr, rl, p, nor, p)
    assert max(relerr(val[r], o.eval(den[r])) for r in range(nrhs)) <= PARITY
    m = f.eval(den, nrhs=nrhs, mode=K.MODE_MIXED).reshape(nrhs, -1)
    assert max(relerr(m[r], val[r]) for r in range(nrhs)) <= MIXED_VS_PLAIN
