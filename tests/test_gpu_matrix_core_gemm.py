"""GPU: the matrix-core GEMMs of the mixed passes and of the transposed FP64 passes,
over the launch sizes where their kernel changes (chunk-splitting strips, 16 x 8
strips, 32 x 16 strips, 160 x 64 tiles).

All forms run one chain of fused multiply-adds a value, so the same densities give
the same bits whatever the launch size: a pass of several right-hand sides, whose
launches have that many times the columns, must equal the one-RHS pass exactly.  The
transposed pass, which runs on these kernels in the FP64 mode too, is pinned to the
forward one (in FP64 itself pinned to the oracle) at the bars it has elsewhere.
"""
import numpy as np
import pytest

import kifmm
from kifmm import workloads as W
from test_gpu_adjoint import dual_gap

pytestmark = pytest.mark.gpu


# Rows and depths that no row block, step of four or stage of 64 terms divides (26,
# 98, 218 samples), two-part columns, K-chunks fewer and more than a workgroup's
# waves, one column.
@pytest.mark.parametrize("kt,coefs,np_,n,pts", [(111, [1.0, 0.25], 3, 700, 8), (111, [1.0, 0.25], 5, 9000, 10),
                                                (111, [1.0, 0.25], 7, 2500, 60), (321, [1.0, 0.25], 4, 3000, 20),
                                                (511, [1.0, 0.3], 3, 5000, 12)])
def test_gemm_forms(kt, coefs, np_, n, pts):
    pos, nor = W.spheres(n, 740 + n, nsph=5)
    den = np.random.default_rng(741 + n).standard_normal((24, n * (4 if kt in (321, 511) else 1)))
    for prec in ("fp64", "mixed"):
        f = kifmm.FMM3d(kt, coefs, np_, pts, 30, precision=prec)
        f.set_points(pos, nor)
        f.setup()
        den = den[:, :n * f.src_dof]
        if prec == "fp64":
            assert dual_gap(f, 742) < (1e-12 if np_ <= 4 else 1e-10)
        else:
            for nrhs in (2, 24):
                multi = f.evaluate_multi(den[:nrhs])
                for r in (0, nrhs - 1):
                    assert np.array_equal(multi[r], f.evaluate(den[r]))
            assert dual_gap(f, 743) < 1e-5
