"""GPU: the mixed scalar V list on the matrix cores, over the tile forms of its group
lists, against the FP64 mode (itself pinned to the oracle) and the transposed pass.

A wrong or missing product shows at the size of a V-list term (1e-2 and more of the
value); what mixed precision itself leaves is the FP32 rounding of spectra and near
field, which the other mixed tests hold to 1e-6 at these expansion orders.
"""
import numpy as np
import pytest

import kifmm
from kifmm import workloads as W
from test_gpu_adjoint import dual_gap
from test_gpu_parity import rel

pytestmark = pytest.mark.gpu


# One tile of a few groups; levels that end inside a tile; a tile closed by its
# colleagues (thin, scattered lists); frequency counts of every order; separate
# targets; more than four rounds of workgroups; several right-hand sides.
@pytest.mark.parametrize("gen,np_,n,pts,nrhs", [("uniform", 4, 300, 8, 1), ("uniform", 3, 20000, 10, 3),
                                                ("gaussians", 5, 30000, 12, 1), ("spheres", 6, 30000, 20, 2),
                                                ("separate", 4, 9000, 20, 1), ("uniform", 6, 300000, 60, 1)])
def test_tile_forms(gen, np_, n, pts, nrhs):
    tpos = None
    if gen == "spheres":
        pos = W.spheres(n, 750, nsph=6)[0]
    elif gen == "gaussians":
        pos = W.gaussians(n, 751)
    else:
        pos = W.uniform(n, 752)
        if gen == "separate":
            tpos = W.gaussians(7000, 753)
    den = np.random.default_rng(754).standard_normal((nrhs, n))
    val = {}
    for prec in ("fp64", "mixed"):
        f = kifmm.FMM3d(111, [1.0, 0.25], np_, pts, 30, precision=prec)
        f.set_points(pos, None, tpos)
        f.setup()
        val[prec] = f.evaluate(den[nrhs - 1])
    if nrhs > 1:
        assert np.array_equal(f.evaluate_multi(den)[nrhs - 1], val["mixed"])
    assert dual_gap(f, 755) < 1e-5
    assert rel(val["mixed"], val["fp64"]) < 1e-5


# The two kernels of the mixed scalar V list give the same bits.  A launch of up to four
# rounds of 512 workgroups (tiles of up to 32 groups x H / 8 frequencies x right-hand
# sides) takes the matrix cores, a larger one whose tiles are not filled (24 groups a
# tile) the vector unit's sweep.  Few groups on every level: at most a tile for five of
# them (a tile holds 144 colleagues, a group has 26), so that one right-hand side surely
# takes the former; at least a tile a level, so that many surely take the latter.
@pytest.mark.parametrize("np_,nrhs,n,pts", [(4, 64, 300, 20), (6, 24, 300, 20), (8, 9, 900, 40), (6, 12, 700, 20)])
def test_both_kernels_same_bits(np_, nrhs, n, pts):
    H = (4 * np_ ** 3 + 4 + 15) // 16 * 16
    if n == 700:  # a clustered tree: a few groups on each of several levels
        pos = 0.37 + 0.6 * np.random.default_rng(756).random((n, 3)) ** 6
    else:
        pos = W.uniform(n, 757)
    f = kifmm.FMM3d(111, [1.0, 0.25], np_, pts, 30, precision="mixed")
    f.set_points(pos)
    f.setup()
    t = f.tree()
    off = t["lists"]["v"][0]
    groups = {(int(t["depth"][b]), int(t["parent"][b])) for b in range(len(off) - 1) if off[b + 1] > off[b]}
    levels = np.bincount([d for d, _ in groups])
    levels = levels[levels > 0]
    print("groups a level", levels, flush=True)
    assert ((levels + 4) // 5).sum() * (H // 8) <= 4 * 512
    assert levels.sum() < 24 * len(levels) and len(levels) * (H // 8) * nrhs > 4 * 512
    den = np.random.default_rng(758).standard_normal((nrhs, n))
    multi = f.evaluate_multi(den)
    for r in (0, nrhs // 2, nrhs - 1):
        assert np.array_equal(multi[r], f.evaluate(den[r]))
