"""The two launch shapes of the tiled matrix-core M2L in the plain form: pinned,
form 0 runs one block per tile and form 4 one wave per tile and frequency, the
same products in another order (fmm3d/fmm3d_eval.cpp:115-150).

Both against the oracle at the parity bar: a uniform tree whose tiles have
every halo parent and a clustered one with absent children, one and two groups
of 16 right-hand sides.  Between the two only the order of a sum of 189 complex
products per output and its rounding differ (378 2^-53, 4e-14); that the results
differ at all shows that two kernels ran.  The last case's 32,768 level-5
sources hold 8.5 GB of spectra, past what 32-bit halo offsets reach.
"""
import numpy as np
import pytest

import kifmm3d as K
from problems import clusters, densities, relerr, uniform_cube
from test_gpu_parity import PARITY, make_fmm, make_oracle

pytestmark = pytest.mark.gpu


def both(f, den, nrhs):
    nlev = len(f.settings(K.MODE_PLAIN)["m2l"])
    out = {}
    for form in (0, 4):
        f.set_settings(K.MODE_PLAIN, -1, [form] * nlev)
        assert f.settings(K.MODE_PLAIN)["m2l"] == [form] * nlev
        out[form] = f.eval(den, nrhs=nrhs).reshape(nrhs, -1).copy()
        assert np.all(np.isfinite(out[form]))
    assert not np.array_equal(out[0], out[4])
    worst = max(relerr(out[0][r], out[4][r]) for r in range(nrhs))
    print(f"  {nlev} levels, block per tile against wave per tile {worst:.3e}", flush=True)
    assert worst <= 1e-13
    return out


@pytest.mark.parametrize("geom,np_,n,nrhs", [("cube", 4, 3000, 16), ("clusters", 4, 4000, 32), ("cube", 6, 9000, 32),
                                             ("clusters", 8, 3000, 16)])
def test_block_and_wave_per_tile_against_the_oracle(geom, np_, n, nrhs):
    print(f"\n[case] {geom} np={np_} n={n} nrhs={nrhs}", flush=True)
    p = (uniform_cube if geom == "cube" else clusters)(n, 31)
    f = make_fmm(111, np_, 30, 10, (0.5, 0.5, 0.5), 1, p, None, p)
    den = densities(n, 1, nrhs, 32)
    nlev = len(f.settings(K.MODE_PLAIN)["m2l"])
    assert f.settings(K.MODE_PLAIN)["m2l"] == [0] * nlev
    default = f.eval(den, nrhs=nrhs).reshape(nrhs, -1).copy()
    assert f.settings(K.MODE_PLAIN)["m2l"] == [4] * nlev  # what the evaluate ran
    out = both(f, den, nrhs)
    assert np.array_equal(default, out[4])
    o = make_oracle(f, 111, np_, 30, 10, (0.5, 0.5, 0.5), 1, p, None, p)
    for r in (0, nrhs - 1):
        ref = o.eval(den[r])
        assert relerr(out[0][r], ref) <= PARITY and relerr(out[4][r], ref) <= PARITY


def test_halo_offsets_beyond_32_bits():
    n, nrhs = 400000, 16
    print(f"\n[case] cube np=6 n={n} nrhs={nrhs}", flush=True)
    p = uniform_cube(n, 33)
    f = make_fmm(111, 6, 30, 10, (0.5, 0.5, 0.5), 1, p, None, p)
    assert f.info()["sndecnt"] > 32768
    both(f, densities(n, 1, nrhs, 34), nrhs)
