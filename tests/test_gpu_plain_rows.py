"""Kernels of the plain (materialised rows) path against plain PyTorch sums
of the same terms.  Tolerance: FP64 sums of at most a few hundred terms of
both signs in another order, 1e-13 of the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a - b).norm() / b.norm())


# ten components per pass, two passes per turn; four atoms per workgroup
@pytest.mark.parametrize("n,nb", [(1, 1), (3, 9), (4, 10), (5, 11), (7, 20), (129, 21), (64, 30), (33, 55), (2, 400)])
def test_voigt_contract(n, nb):
    from pyxtal_ff_amd import so4
    g = torch.Generator().manual_seed(n + 1000 * nb)
    beta = torch.randn((n, nb), dtype=torch.float64, generator=g)
    rv = torch.randn((n, nb, 6), dtype=torch.float64, generator=g)
    ref = -(beta.unsqueeze(2) * rv).sum(1)
    out = so4.voigt_contract(beta.cuda(), rv.cuda()).cpu()
    assert out.shape == (n, 6) and _rel(out, ref) < 1e-13
    # operands off the natural layout are copied first
    bt = beta.t().contiguous().cuda().t()
    assert torch.equal(so4.voigt_contract(bt, rv.cuda()).cpu(), out)
