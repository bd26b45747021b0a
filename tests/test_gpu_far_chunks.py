"""Leaves whose lists are long enough to be cut into chunks of 16 and 32 targets:
near field and L2T / M2T over hundreds of entries (fmm3d/fmm3d_eval.cpp:97-113,
:152-176, :211-219), every near-field kernel, against the oracle at the FP64
parity bar; the mixed form, whose FP32 kernels keep the whole chunks, against
the plain one at its own bar.
"""
import pytest

import kifmm3d as K
from problems import densities, relerr
from test_chunk_plan import CUT, sheet
from test_gpu_parity import PARITY, make_fmm, make_oracle

pytestmark = pytest.mark.gpu

MIXED_VS_PLAIN = 1e-6


@pytest.mark.parametrize("cut", range(len(CUT)))
@pytest.mark.parametrize("kt,nrhs", [(111, 1), (111, 21), (311, 2)])
def test_narrow_chunks(cut, kt, nrhs):
    np_, ptsmax, ns, nt, gap, which, width = CUT[cut]
    print(f"\n[case] kt={kt} nrhs={nrhs} {which} lists, width {width}", flush=True)
    src, trg = sheet(ns, nt, 3, gap)
    f = make_fmm(kt, np_, ptsmax, 10, (0.5, 0.5, 0.5), 1, src, None, trg)
    st = f.plan_stats()
    assert st[f"{which}_chunks_fp64"] > st[f"{which}_chunks"]
    den = densities(ns, f.knl.sdof(), nrhs, 3)
    o = make_oracle(f, kt, np_, ptsmax, 10, (0.5, 0.5, 0.5), 1, src, None, trg)
    ref = {r: o.eval(den[r]) for r in {0, nrhs - 1}}
    for near in (0, 1, 2) if kt == 111 else (0, 1):
        f.set_settings(K.MODE_PLAIN, near)
        val = f.eval(den, nrhs=nrhs).reshape(nrhs, -1).copy()
        for r in ref:
            assert relerr(val[r], ref[r]) <= PARITY
        print(f"  near {near}: {f.kernel_times()['p2p'][0] * 1e3:.1f} us", flush=True)
    m = f.eval(den, nrhs=nrhs, mode=K.MODE_MIXED).reshape(nrhs, -1)
    assert max(relerr(m[r], val[r]) for r in range(nrhs)) <= MIXED_VS_PLAIN
