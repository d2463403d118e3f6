"""GPU: the FP64 kernels that keep the reference's summation order, at the sizes
where their launch forms change, against the CPU oracle.

The bound is the parity bar of the FP64 path (relative 2-norm 1e-12): the level
GEMMs and the V-list sums form the same terms in the same order as the oracle, so
what is left are the near field's rounding and the 1e-16 of each output.
"""
import numpy as np
import pytest

import oracle as O
from kifmm import workloads as W
from test_gpu_parity import PARITY, rel, run_pair

pytestmark = pytest.mark.gpu


# Level GEMMs: one, two and four columns a lane in strips of 16 rows, whole columns
# a lane; row counts that no strip or row set divides (26, 98, 104, 150), depths
# that no slab does (98, 208, 294, 832), one column (the root's children's parent).
@pytest.mark.parametrize("kt,coefs,np_,n,pts", [(111, [1.0, 0.25], 3, 500, 8), (111, [1.0, 0.25], 4, 60000, 6),
                                                (311, [1.0, 0.25], 3, 20000, 10), (511, [1.0, 0.3], 5, 3000, 20),
                                                (111, [1.0, 0.25], 6, 30000, 20)])
def test_level_gemm_forms(kt, coefs, np_, n, pts):
    pos = W.uniform(n, 700 + n)
    den = W.densities(n, O.src_dof(kt), 701 + n, kind="normal")
    _, val, ref = run_pair(kt, coefs, np_, pts, pos, np.zeros_like(pos), den)
    assert rel(val, ref) <= PARITY


# V-list sums: frequency counts that are no multiple of a chunk (np 5: 600), factors
# 1/G that are powers of two (np 4, 8) and not, lists of very different lengths,
# a few groups and more than a pass of a workgroup.
@pytest.mark.parametrize("kt,coefs,np_,n,pts", [(111, [1.0, 0.25], 5, 12000, 10), (111, [1.0, 0.25], 7, 6000, 40),
                                                (111, [1.0, 0.25], 8, 4000, 60), (321, [1.0, 0.25], 5, 2500, 20),
                                                (511, [1.0, 0.3], 3, 6000, 8)])
def test_vlist_forms(kt, coefs, np_, n, pts):
    pos = W.gaussians(n, 710 + n)
    nor = np.random.default_rng(711 + n).standard_normal((n, 3))
    nor /= np.linalg.norm(nor, axis=1)[:, None]
    den = W.densities(n, O.src_dof(kt), 712 + n, kind="normal")
    _, val, ref = run_pair(kt, coefs, np_, pts, pos, nor, den, max_level=12)
    assert rel(val, ref) <= PARITY


# Near field: chunks of one point, of odd counts, of whole 128-point rounds and just
# above; blocks that end inside an item; more items than a staging window (thin
# leaves beside coarse ones); separate targets; pairs under the 1e-8 cut.
@pytest.mark.parametrize("kt", [111, 121, 311, 322, 521])
@pytest.mark.parametrize("n,pts,gen", [(9, 4, "uniform"), (1040, 131, "uniform"), (2100, 300, "uniform"),
                                       (6000, 3, "gauss"), (3000, 500, "close")])
def test_near_forms(kt, n, pts, gen):
    rng = np.random.default_rng(720 + n)
    if gen == "gauss":
        pos = W.gaussians(n, 721, ng=2, smin=0.002, smax=0.02)
    else:
        pos = W.uniform(n, 722 + n)
    if gen == "close":
        pos[1::7] = np.minimum(pos[::7][:len(pos[1::7])] + 3e-9, W.HI)
    nor = rng.standard_normal((n, 3))
    nor /= np.linalg.norm(nor, axis=1)[:, None]
    tpos = W.uniform(n // 2 + 1, 723) if gen == "uniform" else None
    den = rng.standard_normal(n * O.src_dof(kt))
    _, val, ref = run_pair(kt, [1.0, 0.3], 3, pts, pos, nor, den, max_level=16, tpos=tpos)
    assert rel(val, ref) <= PARITY
