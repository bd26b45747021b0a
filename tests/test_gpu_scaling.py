"""The plain form is linear: densities scaled by a power of two give values scaled
by it, bit for bit, as long as no quantity of the algorithm itself leaves the
FP64 range (fmm3d/fmm3d_eval.cpp:24-243).  The pseudoinverse applies, whose
products pass their results by several powers of ten, must not narrow that range.
"""
import numpy as np
import pytest

import kifmm3d as K
from problems import clusters, densities, sphere, uniform_cube
from test_gpu_parity import make_fmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kt,np_,geom,n,nrhs", [(111, 4, "cube", 3000, 1), (111, 6, "clusters", 4000, 16),
                                                (111, 8, "cube", 4000, 2), (521, 6, "sphere", 3000, 1),
                                                (511, 8, "clusters", 2500, 1)])
def test_values_scale_with_the_densities(kt, np_, geom, n, nrhs):
    print(f"\n[case] kt={kt} np={np_} {geom} n={n} nrhs={nrhs}", flush=True)
    p, nor = sphere(n, 71) if geom == "sphere" else ((uniform_cube if geom == "cube" else clusters)(n, 71), None)
    ctr, lvl = ((0.0, 0.0, 0.0), 0) if geom == "sphere" else ((0.5, 0.5, 0.5), 1)
    f = make_fmm(kt, np_, 60, 10, ctr, lvl, p, nor, p)
    den = densities(n, f.knl.sdof(), nrhs, 72)
    ref = f.eval(den, nrhs=nrhs).copy()
    # the largest equivalent density and its level scale leave 2^30 for the M2L sums and the sums over points
    top = 1023 - 30 - int(np.ceil(np.log2(max(np.abs(f.buffer(b)).max() for b in range(4)) + np.abs(ref).max())))
    for k in (-850, -400, 700, top):
        val = f.eval(np.ldexp(den, k), nrhs=nrhs)
        assert np.array_equal(val, np.ldexp(ref, k)), k
    print(f"  2^-850 to 2^{top}", flush=True)
