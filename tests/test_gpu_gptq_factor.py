"""The GPTQ factor of a permuted, damped Hessian (amct_gptq_factor) against the reference's three factorisations
(gptq_module.py:108-121) in fp64."""
import pytest
import torch

from amct_amd import ops

pytestmark = pytest.mark.gpu


# one column, the edges of the 64-column steps, a last step of one column, many steps
@pytest.mark.parametrize("cols", [1, 63, 64, 65, 128, 200, 1099, 2817])
def test_factor(dev, cols):
    g = torch.Generator().manual_seed(cols)
    x = torch.randn(2 * cols + 8, cols, generator=g) * (1 + 5 * (torch.arange(cols) % 37 == 3))
    if cols > 4:
        x[:, 4] = 0                                                # a dead channel: zero row, column and diagonal
    h = (x.t() @ x) * (2.0 / x.shape[0])
    d = torch.diag(h)
    hd = h.double()
    hd[d == 0, d == 0] = 1
    perm = torch.argsort(torch.diag(hd), descending=True)
    damp = (0.01 * torch.diag(hd).mean()).float()
    hp = hd[perm][:, perm] + damp.double() * torch.eye(cols, dtype=torch.float64)
    want = torch.linalg.cholesky(torch.cholesky_inverse(torch.linalg.cholesky(hp)), upper=True)
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    got = ops.gptq_factor(h.to(dev), perm.to(dev), damp.to(dev), bad).cpu().double()
    assert int(bad) == 0
    assert torch.equal(got, torch.triu(got)), "zeros below the diagonal"
    # a Cholesky factorisation of n columns is exact for a matrix within (n + 1) u of its entries (u = 2^-24), which moves
    # the inverse factor by at most that times the condition number; the inverse adds as much again
    ev = torch.linalg.eigvalsh(hp)
    bound = 2 * (cols + 1) * 2.0 ** -24 * float(ev[-1] / ev[0])
    assert float((got - want).norm() / want.norm()) <= bound
    # u hp u^T = I, which the third factorisation does not enter
    assert float((got @ hp @ got.t() - torch.eye(cols, dtype=torch.float64)).abs().max()) <= bound * cols ** 0.5


def test_factor_of_an_indefinite_matrix_is_reported(dev):
    h = torch.eye(100)
    h[40, 41] = h[41, 40] = 3.0
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    ops.gptq_factor(h.to(dev), torch.arange(100, device=dev), torch.zeros((), device=dev), bad)
    assert int(bad) == 1
