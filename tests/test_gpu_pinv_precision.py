"""The compensated pseudoinverse applies of the plain form hold the precision of
a compensated dot product on every operator, np 8 vector kernels included.

upeden = UC2UE upcval (fmm3d/matmgnt3d.cpp:91-123) and dneden = DC2DE dncval
(:158-188), up to the power-of-two level scale of each degree of freedom,
against exact dot products: every product is split into its rounded value and
its error (Dekker), and math.fsum adds the parts with one rounding.

Tolerance: half a unit in the last place of the exact value, and the error of
hi + lo before that rounding, in units of 2^-106.  For K < 256 that is the bound
of Dot2 (Ogita, Rump and Oishi 2005), K^2 sum |a b|.  Otherwise, with n = K / 8
blocks of 8 products, S the sum over the blocks of (sum of |a|) (max of |b|) and
R the largest partial sum: a block's running sum stays below 3 times its S, so
the 8 rests are at most 3 2^-53 S each, their roundings 24 S, those of the 7
additions of the rests 78 S, of adding their sum to the running one at most 48 S
more, together under 160 S; and lo, at most 2^-53 j R after j blocks (2 R in a
part of K), is rounded n times, (n + 2)^2 / 2 R.
"""
import math

import numpy as np
import pytest

import kifmm3d as K
from problems import COEFS, clusters, densities, sphere, uniform_cube

pytestmark = pytest.mark.gpu


def _split(a):
    c = 134217729.0 * a  # 2^27 + 1
    hi = c - (c - a)
    return hi, a - hi


def _exact_dots(A, x):
    p = A * x
    ah, al = _split(A)
    xh, xl = _split(x)
    e = ((ah * xh - p) + ah * xl + al * xh) + al * xl
    return np.array([math.fsum(r) for r in np.concatenate([p, e], axis=1)]), p


def _bound(A, x, p):
    k = A.shape[1]
    if k < 256:
        return 2.0 ** -106 * k * k * np.abs(p).sum(axis=1)
    s = np.abs(A).reshape(len(A), -1, 8).sum(axis=2) @ np.abs(x).reshape(-1, 8).max(axis=1)
    r = np.abs(np.cumsum(p, axis=1)).max(axis=1)
    return 2.0 ** -106 * (160 * s + 0.5 * (k // 8 + 2) ** 2 * r)


@pytest.mark.parametrize("kt,np_,geom,n,ptsmax,nrhs,nodes,step", [
    (311, 8, "clusters", 4000, 60, 1, 24, 1), (111, 8, "cube", 9001, 60, 5, 24, 3), (521, 6, "sphere", 9000, 60, 1, 16, 3),
    (111, 6, "cube", 60000, 30, 16, 16, 3), (511, 4, "clusters", 4001, 40, 3, 24, 3), (111, 4, "cube", 2999, 40, 1, 24, 1)])
def test_pinv_applies_to_twice_working_precision(kt, np_, geom, n, ptsmax, nrhs, nodes, step):
    print(f"\n[case] kt={kt} np={np_} {geom} n={n} ptsmax={ptsmax} nrhs={nrhs}", flush=True)
    pos, nor = sphere(n, 21) if geom == "sphere" else ((uniform_cube if geom == "cube" else clusters)(n, 21), None)
    f = K.FMM3d("fmm3d_")
    f.srcpos, f.srcnor, f.trgpos = pos, nor, pos
    f.ctr, f.rootlvl = ((0.0, 0.0, 0.0), 0) if geom == "sphere" else ((0.5, 0.5, 0.5), 1)
    f.knl = K.Kernel3d(kt, COEFS[kt])
    f.setup({"-fmm3d_np": str(np_), "-fmm3d_let3d_ptsmax": str(ptsmax), "-fmm3d_let3d_maxlevel": "10"})
    f.eval(densities(n, f.knl.sdof(), nrhs, 3), nrhs=nrhs)
    dof = {111: 1, 511: 3, 521: 3}.get(kt, 4)  # of the translation kernel's densities
    rng = np.random.default_rng(5)
    for op, den, chk in ((0, 0, 1), (1, 2, 3)):
        P = f.operator(op)
        m, k = P.shape
        y, x = f.buffer(den).reshape(-1, m), f.buffer(chk).reshape(-1, k)
        live = np.flatnonzero(np.any(y != 0, axis=1) & np.any(x != 0, axis=1))
        off = tot = 0
        for g in rng.choice(live, min(nodes, live.size), replace=False):
            rows = np.arange(int(rng.integers(0, step)), m, step)
            ex, p = _exact_dots(P[rows], x[g])
            tol = 2.0 ** -53 * np.abs(ex) * (1 + 2.0 ** -40) + _bound(P[rows], x[g], p)
            for d in range(dof):
                sel = (rows % dof == d) & (ex != 0)
                scale = 2.0 ** np.round(np.median(np.log2(np.abs(y[g][rows[sel]] / ex[sel]))))
                off += int(np.sum(np.abs(y[g][rows[sel]] / scale - ex[sel]) > tol[sel]))
                tot += int(sel.sum())
        print(f"  operator {op} ({m} x {k}): {off} of {tot} results outside", flush=True)
        assert off == 0
