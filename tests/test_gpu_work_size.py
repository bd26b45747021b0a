"""The work memory of an evaluate has no split-K partials for products whose
splits are summed within a block: 16 x columns x operator rows doubles, 117 MB
for this problem's 1,536 Stokes boxes at np 6, beside 215 MB for all the rest.
The no-allocation evaluate, whose array holds 256 MiB, takes the problem, and
gives the bits of the ordinary one.
"""
import numpy as np
import pytest

import kifmm3d as K
from problems import COEFS, densities

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [K.MODE_PLAIN, K.MODE_MIXED])
def test_no_alloc_without_split_partials(mode):
    n = 15000
    print(f"\n[case] noalloc stokes n={n} np=6 mode={mode}", flush=True)
    p = np.random.default_rng(61).random((n, 3)) * np.array([1.0, 1.0, 0.37])
    f = K.FMM3d("fmm3d_")
    f.srcpos, f.srcnor, f.trgpos = p, None, p
    f.ctr, f.rootlvl = (0.5, 0.5, 0.5), 1
    f.knl = K.Kernel3d(311, COEFS[311])
    f.setup({"-fmm3d_np": "6", "-fmm3d_let3d_ptsmax": "40", "-fmm3d_let3d_maxlevel": "10"})
    assert f.info()["sndecnt"] > 1536
    den = densities(n, 3, 1, 62)
    src, ref, got = (K.DeviceBuffer(n * 3 * 8) for _ in range(3))
    src.upload(den)
    got.upload(np.full(n * 3, np.nan))
    f.eval_device(src, ref, 1, mode)
    rc = K.lib().kifmm3d_evaluate_device_noalloc(f.h, src.ptr, got.ptr, 1, mode)
    assert rc == K.OK, K.lib().kifmm3d_last_error(f.h)
    a, b = np.empty(n * 3), np.empty(n * 3)
    ref.download(a)
    got.download(b)
    assert np.array_equal(a, b)
