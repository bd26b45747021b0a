"""A target at the origin of the coordinates, the centre of a domain about it: the
FP64 matrix-core near field (blocks of 16 right-hand sides) pads its source
tiles to a multiple of 4 with sources of zero density, which must not lie where
a target can (kernel3d.cpp:21, r < 1e-8, is not tested between far-enough leaves).
"""
import numpy as np
import pytest

import kifmm3d as K
from problems import densities, relerr
from test_gpu_parity import PARITY, make_fmm, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrhs", [16, 21])
@pytest.mark.parametrize("n", [1501, 3000])
def test_target_at_the_origin(n, nrhs):
    print(f"\n[case] n={n} nrhs={nrhs}", flush=True)
    rng = np.random.default_rng(41)
    src = rng.uniform(-1, 1, (n, 3))
    trg = np.concatenate([np.zeros((1, 3)), rng.uniform(-1, 1, (200, 3))])
    f = make_fmm(111, 4, 60, 10, (0.0, 0.0, 0.0), 0, src, None, trg)
    f.set_settings(K.MODE_PLAIN, 2)
    den = densities(n, 1, nrhs, 42)
    val = f.eval(den, nrhs=nrhs).reshape(nrhs, -1).copy()
    assert np.all(np.isfinite(val))
    o = make_oracle(f, 111, 4, 60, 10, (0.0, 0.0, 0.0), 0, src, None, trg)
    for r in (0, nrhs - 1):
        assert relerr(val[r], o.eval(den[r])) <= PARITY
    mixed = f.eval(den, nrhs=nrhs, mode=K.MODE_MIXED).reshape(nrhs, -1)
    assert max(relerr(mixed[r], val[r]) for r in range(nrhs)) <= 1e-6
