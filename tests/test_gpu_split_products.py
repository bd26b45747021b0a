"""Uncompensated products with K split over the waves of a 32 x 32 tile, where a
level has few columns, against the wide-tile kernel with the same splits
(KIFMM3D_GEMM=wide): the same operations in the same order, so both forms'
results agree to the bit, and the plain form's with the oracle at the parity
bar.  Operator rows that leave part of a 32-row tile (56, 152, 168, 456), 1 to
several hundred columns that leave part of a 32-column one, absent children,
two source buffers and accumulation (mixed form).
"""
import numpy as np
import pytest

import kifmm3d as K
from problems import clusters, densities, relerr, sphere
from test_gpu_parity import PARITY, make_fmm, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kt,np_,n,nrhs", [(111, 4, 2500, 1), (111, 4, 2500, 19), (111, 6, 3000, 3),
                                           (321, 6, 2500, 1), (511, 4, 3000, 2)])
def test_split_against_wide(kt, np_, n, nrhs, monkeypatch):
    print(f"\n[case] kt={kt} np={np_} n={n} nrhs={nrhs}", flush=True)
    p, nor = sphere(n, 51) if kt == 321 else (clusters(n, 52), None)
    ctr, rl = ((0.0, 0.0, 0.0), 0) if kt == 321 else ((0.5, 0.5, 0.5), 1)
    out = {}
    for gemm in ("", "wide"):
        if gemm:
            monkeypatch.setenv("KIFMM3D_GEMM", gemm)
        f = make_fmm(kt, np_, 40, 10, ctr, rl, p, nor, p)
        den = densities(n, f.knl.sdof(), nrhs, 53)
        for mode in (K.MODE_PLAIN, K.MODE_MIXED):
            out[gemm, mode] = f.eval(den, nrhs=nrhs, mode=mode).reshape(nrhs, -1).copy()
    for mode in (K.MODE_PLAIN, K.MODE_MIXED):
        assert np.array_equal(out["", mode], out["wide", mode])
    o = make_oracle(f, kt, np_, 40, 10, ctr, rl, p, nor, p)
    for r in range(nrhs):
        assert relerr(out["", K.MODE_PLAIN][r], o.eval(den[r])) <= PARITY
