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
