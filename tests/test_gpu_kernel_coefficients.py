"""GPU: the FP64 pair sums of the Navier kernels at coefficients where one of their
constants vanishes: A of the double layer (521) at nu = 1/2, the incompressible limit
(A = -(1 - 2 nu) / (8 pi (1 - nu))), and G of the single layer (511) at nu = 3/4
(G = (3 - 4 nu) / (16 pi (1 - nu))); nu = 0.3 beside them.

Bars: relative 2-norm 1e-12 against the oracle (the FP64 parity bar); the duality gap
of the transposed pass at the bars it has for the other coefficients.
"""
import numpy as np
import pytest

import kifmm
import oracle as O
from kifmm import workloads as W
from test_gpu_adjoint import dual_gap
from test_gpu_parity import PARITY, rel, run_pair

pytestmark = pytest.mark.gpu

COEFS = [(521, 0.5), (521, 0.3), (511, 0.75), (511, 0.5)]


def problem(kt, n, seed):
    pos, nor = W.spheres(n, seed, nsph=4)
    return pos, nor, W.densities(n, O.src_dof(kt), seed + 1, kind="normal")


@pytest.mark.parametrize("kt,nu", COEFS)
def test_one_box_and_direct(kt, nu):
    """All pairs in one leaf: the near field alone, the direct sum, and the transposed near field."""
    import torch
    n = 301
    pos, nor, den = problem(kt, n, 760)
    print("case one box kt=%d nu=%g" % (kt, nu), flush=True)
    f = kifmm.FMM3d(kt, [1.3, nu], 4, n, 30)
    f.set_points(pos, nor)
    f.setup()
    ref = O.direct(kt, [1.3, nu], pos, nor, den, pos)
    assert rel(f.evaluate(den), ref) <= PARITY
    out = torch.empty(n * f.trg_dof, dtype=torch.float64, device="cuda:0")
    f.direct_device(torch.from_numpy(den).cuda(), torch.from_numpy(pos).cuda(), out)
    assert rel(out.cpu().numpy(), ref) <= PARITY
    assert dual_gap(f, 761) < 1e-12
    if (kt, nu) == (521, 0.5):  # the incompressible double layer is the Stokes one
        assert rel(f.evaluate(den), O.direct(321, [1.0, 0.25], pos, nor, den, pos)) <= PARITY


@pytest.mark.parametrize("kt,nu", [(521, 0.5), (511, 0.5)])
def test_tree(kt, nu):
    pos, nor, den = problem(kt, 3000, 762)
    f, val, ref = run_pair(kt, [1.0, nu], 4, 20, pos, nor, den)
    assert rel(val, ref) <= PARITY
    assert dual_gap(f, 763) < 1e-12
    f = kifmm.FMM3d(kt, [1.0, nu], 4, 20, 30, precision="mixed")
    f.set_points(pos, nor)
    f.setup()
    assert dual_gap(f, 764) < 1e-5
