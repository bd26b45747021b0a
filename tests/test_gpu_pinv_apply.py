"""The compensated pseudoinverse applies of the plain form against exact dot products.

upeden = UC2UE upcval and dneden = DC2DE dncval (fmm3d/matmgnt3d.cpp:91-123,
158-188), up to the power-of-two level scale of each degree of freedom.  The
reference values are exact: every product is split into its rounded value and
its error (Dekker), and math.fsum adds the parts with one rounding.

Tolerance: with u = 2^(m - 52) the unit of the running sum, 2^m <= 8 rowsum
and the column scaled by 2^e <= 2 colmax, the K split-off errors are at most
u / 2 each, so their own sum is off by at most (K + 1)^2 2^-54 u; plus half a
unit in the last place of the result.
"""
import math

import numpy as np
import pytest

import kifmm3d as K
from problems import COEFS, densities, uniform_cube

pytestmark = pytest.mark.gpu


def _split(a):
    c = 134217729.0 * a  # 2^27 + 1
    hi = c - (c - a)
    return hi, a - hi


def _exact_dot(a, b):
    p = a * b
    ah, al = _split(a)
    bh, bl = _split(b)
    e = ((ah * bh - p) + ah * bl + al * bh) + al * bl
    return math.fsum(np.concatenate([p, e]))


# column counts of every split of K: 16, 8 and 4 waves a tile, one wave a tile
# (scales by their own pass in the last two), with ragged tiles
@pytest.mark.parametrize("kt,np_,n,ptsmax,nrhs", [
    (111, 4, 2999, 40, 1), (111, 6, 20000, 60, 16), (111, 8, 9001, 60, 5), (311, 4, 20000, 60, 3),
    (311, 6, 30011, 60, 1), (111, 6, 60000, 30, 16)])
def test_pinv_applies_are_exact_to_one_rounding(kt, np_, n, ptsmax, nrhs):
    print(f"\n[case] kt={kt} np={np_} n={n} ptsmax={ptsmax} nrhs={nrhs}", flush=True)
    pos = uniform_cube(n, 11)
    f = K.FMM3d("fmm3d_")
    f.srcpos, f.srcnor, f.trgpos = pos, pos, pos
    f.ctr, f.rootlvl = (0.5, 0.5, 0.5), 1
    f.knl = K.Kernel3d(kt, COEFS[kt])
    f.setup({"-fmm3d_np": str(np_), "-fmm3d_let3d_ptsmax": str(ptsmax), "-fmm3d_let3d_maxlevel": "10"})
    f.eval(densities(n, f.knl.sdof(), nrhs, 3), nrhs=nrhs)
    dof = 1 if kt == 111 else 4  # of the translation kernel's densities
    rng = np.random.default_rng(5)
    worst = 0.0
    for op, den, chk in ((0, 0, 1), (1, 2, 3)):
        P = f.operator(op)
        m, k = P.shape
        y, x = f.buffer(den).reshape(-1, m), f.buffer(chk).reshape(-1, k)
        rows = np.abs(P).sum(axis=1)
        nodes = np.flatnonzero(np.any(y != 0, axis=1) & np.any(x != 0, axis=1))
        assert nodes.size >= 64
        for g in rng.choice(nodes, 24, replace=False):
            pick = np.concatenate([[0, m - 1], rng.integers(0, m, 30)])
            ex = np.array([_exact_dot(P[i], x[g]) for i in pick])
            for d in range(dof):
                sel = np.flatnonzero((pick % dof == d) & (ex != 0))
                if sel.size == 0:
                    continue
                scale = 2.0 ** np.round(np.median(np.log2(np.abs(y[g][pick[sel]] / ex[sel]))))
                err = np.abs(y[g][pick[sel]] / scale - ex[sel])
                tol = 2.0 ** -53 * np.abs(ex[sel]) * (1 + 2.0 ** -40) + \
                    (k + 1) ** 2 * 2.0 ** -106 * 16 * rows[pick[sel]] * np.abs(x[g]).max()
                worst = max(worst, float((err / tol).max()))
    print(f"  largest error / tolerance {worst:.3f}", flush=True)
    assert worst <= 1.0
