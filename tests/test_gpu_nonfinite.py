"""GPU: densities that are not finite, or so large that their spectra may not be, in the
FP64 pass.  The V-list sums take a group's sources without a look at their membership
only if every one's transform input is finite (and below 1e290); otherwise member by
member, so that a source adds nothing to the targets it is adjacent to.

Against the CPU oracle: infinite, NaN and finite values at the same places, the finite
ones within the FP64 parity bar (relative 2-norm 1e-12).
"""
import numpy as np
import pytest

import kifmm
import oracle as O
from kifmm import workloads as W
from test_gpu_adjoint import direct_grad
from test_gpu_parity import PARITY, run_pair

pytestmark = pytest.mark.gpu


def agree(val, ref):
    for what in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(what(val), what(ref)), what.__name__
    fin = np.isfinite(ref)
    print("finite %d of %d, +inf %d, -inf %d" % (fin.sum(), ref.size, np.isposinf(ref).sum(), np.isneginf(ref).sum()),
          flush=True)
    if fin.any():
        big = np.abs(ref[fin]).max()
        d, s = (val[fin] / big) - (ref[fin] / big), ref[fin] / big
        assert np.linalg.norm(d) <= PARITY * np.linalg.norm(s)


# np 4: 1/G a power of two; 5: not, and frequency counts that no chunk divides.  Depth 2
# and more: V lists on several levels; the group of the source, and groups beside it.
@pytest.mark.parametrize("kt,np_,n,pts", [(111, 4, 1500, 8), (111, 5, 300, 8), (311, 4, 500, 12), (511, 5, 300, 12)])
@pytest.mark.parametrize("bad", [np.inf, np.nan, 1e294])
def test_one_bad_density(kt, np_, n, pts, bad):
    coefs = [1.0, 0.3]
    pos = W.uniform(n, 780 + n)
    sd = O.src_dof(kt)
    rng = np.random.default_rng(781)
    den = rng.standard_normal((3, n * sd))
    den[1, (n // 3) * sd] = bad
    f, val, ref = run_pair(kt, coefs, np_, pts, pos, np.zeros_like(pos), den[1])
    agree(val, ref)
    # three right-hand sides, one of them bad: the others are untouched
    multi = f.evaluate_multi(den)
    assert np.array_equal(multi[1], val, equal_nan=True)
    for r in (0, 2):
        assert np.isfinite(multi[r]).all()
        assert np.array_equal(multi[r], f.evaluate(den[r]))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_field_at_the_bad_source(bad, precision):
    """A pair under the 1e-8 cut adds nothing to the gradient, whatever its density: the
    bad source's own point keeps its finite gradient, every other point loses it."""
    n, j = 150, 41
    pos = W.uniform(n, 782)
    den = np.random.default_rng(783).standard_normal(n)
    den[j] = bad
    f = kifmm.FMM3d(111, [1.0, 0.25], 4, n, 30, precision=precision)
    f.set_points(0.5 * pos)
    f.setup()
    g = f.field(den).reshape(n, 3)
    others = np.arange(n) != j
    ref = direct_grad(0.5 * pos[others], den[others], 0.5 * pos[j:j + 1])[0]
    assert np.linalg.norm(g[j] - ref) <= PARITY * np.linalg.norm(ref)
    assert not np.isfinite(g[others]).any()


@pytest.mark.parametrize("kt", [121, 311, 312, 321, 322, 511, 521])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 1e294])
def test_pair_sums(kt, bad):
    """One box 1e-3 wide: near field, direct sum and transposed near field give an infinity
    where the kernel block times the density does, and lose no finite value on the way."""
    import torch
    n, j, coefs = 150, 67, [1.0, 0.3]
    pos = 0.3 + 1e-3 * W.uniform(n, 784)
    rng = np.random.default_rng(785)
    nor = rng.standard_normal((n, 3))
    nor /= np.linalg.norm(nor, axis=1)[:, None]
    f = kifmm.FMM3d(kt, coefs, 4, n, 30)
    f.set_points(pos, nor)
    f.setup()
    den = rng.standard_normal(n * f.src_dof)
    den[j * f.src_dof] = bad
    ref = O.direct(kt, coefs, pos, nor, den, pos)
    val = f.evaluate(den)
    agree(val, ref)
    good = rng.standard_normal((2, den.size))
    multi = f.evaluate_multi(np.stack([good[0], den, good[1]]))
    assert np.array_equal(multi[1], val, equal_nan=True)
    assert np.array_equal(multi[0], f.evaluate(good[0])) and np.array_equal(multi[2], f.evaluate(good[1]))
    out = torch.empty(n * f.trg_dof, dtype=torch.float64, device="cuda:0")
    f.direct_device(torch.from_numpy(den).cuda(), torch.from_numpy(pos).cuda(), out)
    agree(out.cpu().numpy(), ref)
    w = rng.standard_normal(n * f.trg_dof)
    w[j * f.trg_dof] = bad
    M = O.kernel_matrix(kt, coefs, pos, nor, pos)
    with np.errstate(invalid="ignore"):
        agree(f.evaluate_adjoint(w), (M * w[:, None]).sum(0))
