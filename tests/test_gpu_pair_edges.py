"""GPU: the FP64 pair sums at the edges of their range, against the CPU oracle (relative
2-norm 1e-12, the FP64 parity bar) and by the transposed pass.
"""
import numpy as np
import pytest

import kifmm
import oracle as O
from kifmm import workloads as W
from test_gpu_adjoint import dual_gap
from test_gpu_parity import PARITY, rel, run_pair

pytestmark = pytest.mark.gpu


def deep_boxes(n, seed):
    """n points, the first eleven in two boxes of level 27 (7.5e-9 wide): three in a
    leaf, eight in a split one beside it, in the child box that does not touch the
    leaf.  Of that child the leaf sees the equivalent surface, of its own box the
    outer one, both closer than the 1e-8 pair cut in part; its only source list
    entry is itself."""
    pos = W.uniform(n, seed)
    p = np.floor(pos[0] * 2.0 ** 26)
    rng = np.random.default_rng(seed + 1)
    pos[:3] = (2 * p + rng.random((3, 3))) * 2.0 ** -27
    for k in range(8):
        child = 2 * (4 * p + (3, 1, 0)) + (k >> 2, (k >> 1) & 1, k & 1)
        pos[3 + k] = (child + rng.random(3)) * 2.0 ** -29
    return pos


@pytest.mark.parametrize("kt", [111, 121, 311])
def test_surfaces_under_the_pair_cut(kt):
    n = 400
    rng = np.random.default_rng(770)
    pos = deep_boxes(n, 771)
    nor = rng.standard_normal((n, 3))
    nor /= np.linalg.norm(nor, axis=1)[:, None]
    den = rng.standard_normal(n * O.src_dof(kt))
    f, val, ref = run_pair(kt, [1.0, 0.25], 4, 6, pos, nor, den)
    assert f.tree()["max_depth"] == 29
    deep = 3 * O.trg_dof(kt)
    assert np.abs(val[:deep] - ref[:deep]).max() <= 1e-12 * np.abs(ref).max()
    assert rel(val, ref) <= PARITY
    assert dual_gap(f, 772) < 1e-12


@pytest.mark.parametrize("kt", [111, 121, 311, 312, 321, 521])
def test_direct_far_targets(gpu, kt):
    """Check targets so far that r^2 (and earlier its powers) overflow."""
    import torch
    n = 700
    pos, nor = W.spheres(n, 774, nsph=3)
    den = np.random.default_rng(775).standard_normal(n * O.src_dof(kt))
    f = kifmm.FMM3d(kt, [1.0, 0.3], 4, 64, 30)
    f.set_points(pos, nor)
    f.setup()
    chk = np.random.default_rng(776).standard_normal((1030, 3))
    for k, s in enumerate((1e60, 1e100, 1e153, 1.3e154, 1e155, 1e200, 1e300)):
        chk[k::9] *= s
    out = torch.empty(len(chk) * f.trg_dof, dtype=torch.float64, device="cuda:0")
    f.direct_device(torch.from_numpy(den).cuda(), torch.from_numpy(chk).cuda(), out)
    ref = O.direct(kt, [1.0, 0.3], pos, nor, den, chk)
    assert np.isfinite(ref).all()
    out = out.cpu().numpy()
    assert rel(out, ref) <= PARITY
    far = np.abs(np.repeat(chk, f.trg_dof, axis=0)).max(1) > 1e150
    assert np.abs(out[far] - ref[far]).max() <= 1e-140


def test_domain_far_from_the_origin():
    """A domain around (1e18, 0, 0) with a point there, a round place that the padding of
    the packed sources must not have."""
    n = 3000
    c = np.array([1e18, 0.0, 0.0])
    pos = c + 128.0 * np.random.default_rng(777).integers(-2 ** 33, 2 ** 33, (n, 3))
    pos[7] = c
    den = np.random.default_rng(778).standard_normal(n)
    f = kifmm.FMM3d(111, [1.0, 0.25], 3, 40, 4, ctr=c, root_level=-40)
    f.set_points(pos)
    f.setup()
    val = f.evaluate(den)
    assert np.isfinite(val).all()
    ops = O.Ops(111, [1.0, 0.25], 3, f.operator(0).reshape(98, 26).T, f.operator(1).reshape(26, 26).T)
    tree = O.Tree(pos, None, ctr=c, root_level=-40, pts_max=40, max_level=4)
    ref = O.evaluate(tree, ops, 111, [1.0, 0.25], pos, np.zeros_like(pos), pos, den, root_level=-40, ctr=c)
    assert rel(val, ref) <= PARITY
