"""Near field and L2T / M2T over chunks of every shape: lanes and waves that
share a target's sources, tiles that cross the entries of a chunk's list, more
entries than one batch of 64, and leaves cut into chunks of 16 to 128 targets.

A tight cluster beside a sparse cloud makes leaves of 1 to 128 points, lists of
a few to several thousand sources and W boxes by the dozen; targets of their
own put thousands into one leaf.  The plain form is held against the oracle at
the FP64 parity bar, the mixed form against the plain one at its own bar.
"""
import numpy as np
import pytest

import kifmm3d as K
from problems import densities, relerr, sphere, uniform_cube
from test_gpu_parity import PARITY, make_fmm, make_oracle

pytestmark = pytest.mark.gpu

MIXED_VS_PLAIN = 1e-6


def points(n, seed):
    """Four fifths of the points in a ball of radius ~0.005 next to a coarse box, the rest uniform."""
    rng = np.random.default_rng(seed)
    k = n * 4 // 5
    tight = np.array([0.505, 0.3, 0.3]) + 0.002 * rng.standard_normal((k, 3))
    return np.concatenate([tight, uniform_cube(n - k, seed + 1)])


def check(kt, np_, ptsmax, src, nor, trg, nrhs, mixed, ctr=(0.5, 0.5, 0.5), rootlvl=1):
    print(f"\n[case] kt={kt} np={np_} ptsmax={ptsmax} ns={len(src)} nt={len(trg)} nrhs={nrhs}", flush=True)
    f = make_fmm(kt, np_, ptsmax, 10, ctr, rootlvl, src, nor, trg)
    den = densities(len(src), f.knl.sdof(), nrhs, 3)
    val = f.eval(den, nrhs=nrhs).reshape(nrhs, -1).copy()
    o = make_oracle(f, kt, np_, ptsmax, 10, ctr, rootlvl, src, nor, trg)
    for r in sorted({0, nrhs // 2, nrhs - 1}):
        assert relerr(val[r], o.eval(den[r])) <= PARITY
    if mixed:
        m = f.eval(den, nrhs=nrhs, mode=K.MODE_MIXED).reshape(nrhs, -1)
        assert max(relerr(m[r], val[r]) for r in range(nrhs)) <= MIXED_VS_PLAIN
    return f


@pytest.mark.parametrize("kt,nrhs,mixed", [(111, 1, False), (111, 4, False), (111, 21, True), (121, 16, False),
                                           (311, 1, True), (312, 4, False), (511, 5, True), (521, 1, False)])
def test_refined_corner(kt, nrhs, mixed):
    p = points(5000, 11)
    nor = sphere(5000, 12)[1] if kt in (121, 521) else None
    f = check(kt, 4, 40, p, nor, p, nrhs, mixed)
    assert (np.diff(f.list_csr(0)[0]) + np.diff(f.list_csr(2)[0])).max() > 64


@pytest.mark.parametrize("kt,nrhs,mixed", [(111, 1, False), (111, 16, True), (311, 1, False)])
def test_many_targets_in_one_leaf(kt, nrhs, mixed):
    rng = np.random.default_rng(14)
    src = points(3001, 13)
    trg = np.concatenate([rng.uniform(0.9, 0.99, (1500, 3)), uniform_cube(517, 15)])
    check(kt, 4, 60, src, None, trg, nrhs, mixed)


@pytest.mark.parametrize("n", [1, 7, 63, 64, 65, 127, 128, 129, 257])
@pytest.mark.parametrize("nrhs", [1, 16])
def test_single_leaf(n, nrhs):
    p = uniform_cube(n, 16 + n)
    check(111, 4, 300, p, None, p, nrhs, False)
