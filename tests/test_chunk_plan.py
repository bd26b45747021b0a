"""The plan's chunks of targets (CPU): leaves with long lists are cut into
narrower chunks for the FP64 kernels."""
import numpy as np
import pytest

import kifmm3d as K
from problems import uniform_cube


def sheet(ns, nt, seed, gap):
    """Sources on a thin sheet beside the face of a coarse box that holds nt targets, a few everywhere.
    Small gaps put the sheet into the box's U list, larger ones into its W list."""
    rng = np.random.default_rng(seed)
    k = ns * 19 // 20
    src = np.stack([0.5 + gap * (1 + 0.2 * rng.random(k)), rng.uniform(0.25, 0.5, k), rng.uniform(0.25, 0.5, k)], axis=1)
    trg = rng.uniform(0.25, 0.5, (nt, 3))
    return (np.concatenate([src, uniform_cube(ns - k, seed + 1)]), np.concatenate([trg, uniform_cube(200, seed + 2)]))


def host(np_, ptsmax, src, trg):
    f = K.FMM3d("fmm3d_")
    f.srcpos, f.srcnor, f.trgpos = src, None, trg
    f.ctr, f.rootlvl = (0.5, 0.5, 0.5), 1
    f.knl = K.Kernel3d(111, [1.0])
    try:
        f.setup({"-fmm3d_np": str(np_), "-fmm3d_let3d_ptsmax": str(ptsmax), "-fmm3d_let3d_maxlevel": "10"})
    except K.KifmmError as e:
        assert e.code == K.EDEVICE
    return f


# np, ptsmax, sources, targets, gap -> which list is long, and the narrowest width it asks for
CUT = [(4, 150, 9000, 140, 0.002, "near", 16), (4, 100, 20000, 60, 0.02, "far", 16), (4, 150, 6000, 100, 0.04, "far", 32)]


@pytest.mark.parametrize("np_,ptsmax,ns,nt,gap,which,width", CUT)
def test_long_lists_cut_their_leaves(np_, ptsmax, ns, nt, gap, which, width):
    f = host(np_, ptsmax, *sheet(ns, nt, 3, gap))
    st = f.plan_stats()
    assert st["near_chunks_fp64"] >= st["near_chunks"] and st["far_chunks_fp64"] >= st["far_chunks"]
    # the coarse box: one leaf of at least nt targets, in chunks of the width its list asks for
    nodes = f.nodes()
    leaf = max((int(n[12]) for n in nodes if n[1] < 0 and n[6] & 2), default=0)
    extra = st[f"{which}_chunks_fp64"] - st[f"{which}_chunks"]
    assert extra >= -(-leaf // width) - -(-leaf // 128) > 0
