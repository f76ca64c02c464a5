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
    # as far from fp64 as the reference's own sequence in fp32, with room for another order of its sums, tile by tile of the
    # elimination: one wrong tile is far beyond it (half a unit of the largest entry where that sequence is exact)
    h32 = hp.float()
    theirs = torch.linalg.cholesky(torch.cholesky_inverse(torch.linalg.cholesky(h32)), upper=True).double()
    assert float((got - want).norm()) <= 8 * float((theirs - want).norm()) + 2.0 ** -24 * float(want.norm())

    def by_tile(e):
        pad = -cols % 64
        return torch.nn.functional.pad(e, (0, pad, 0, pad)).reshape((cols + pad) // 64, 64, -1, 64).square().sum((1, 3)).sqrt()
    limit = 8 * float(by_tile(theirs - want).max()) + 2.0 ** -24 * float(want.abs().max())
    assert bool((by_tile(got - want) <= limit).all())
    tiles = by_tile(want)
    assert bool((tiles[tiles > 0] > limit).all()), "a lost tile shows (the zeros: the dead channel alone in the last one)"
    # u hp u^T = I, which the third factorisation does not enter
    eye = torch.eye(cols, dtype=torch.float64)
    assert float((got @ hp @ got.t() - eye).abs().max()) <= 8 * float((theirs @ hp @ theirs.t() - eye).abs().max()) + 2.0 ** -22


# rows of the Hessian that come in two pieces (from 16385 columns on) and in five, tile numbers beyond 2^18
@pytest.mark.parametrize("cols", [4160, 16500, 65600])
def test_factor_of_many_columns(dev, cols):
    """The factor of I + V V^T in a random order, without a factorisation to compare with: u is upper triangular and u hp lower
    triangular with the reciprocals of u's diagonal on its own, which only the factor is.  In fp64, some rows at a time."""
    rank, step = 32, 4096
    g = torch.Generator(device=dev).manual_seed(cols)
    v = torch.randn(cols, rank, generator=g, device=dev) / rank ** 0.5
    h = torch.empty(cols, cols, device=dev)
    for i in range(0, cols, step):
        h[i:i + step] = v[i:i + step] @ v.t()
        h[i:i + step, i:i + step].diagonal().add_(1.)
    perm = torch.randperm(cols, generator=g, device=dev)
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    u = ops.gptq_factor(h, perm, torch.full((), 0.0078125, device=dev), bad)
    assert int(bad) == 0
    del h
    v = v[perm].double()
    col = torch.arange(cols, device=dev)
    for i in range(0, cols, step):
        rows = u[i:i + step].double()
        prod = (rows @ v) @ v.t() + 1.0078125 * rows
        at = col[i:i + step, None]
        assert not bool((rows.masked_fill(col >= at, 0) != 0).any()), "zeros below the diagonal"
        # entries of the order of 1 in fp32: 64 units of its rounding, eight times what it measures at each of the sizes; an
        # entry of u far from the diagonal is 5e-5 or more on average, so a lost tile is beyond it
        assert float(prod.masked_fill(col <= at, 0).abs().max()) <= 2.0 ** -18
        diag = rows.gather(1, at) * prod.gather(1, at)
        assert float((diag - 1).abs().max()) <= 2.0 ** -15             # (measured: 4.6e-6 at 65600 columns)
    del u, rows, prod
    torch.cuda.empty_cache()


def test_factor_of_an_indefinite_matrix_is_reported(dev):
    h = torch.eye(100)
    h[40, 41] = h[41, 40] = 3.0
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    ops.gptq_factor(h.to(dev), torch.arange(100, device=dev), torch.zeros((), device=dev), bad)
    assert int(bad) == 1


# one tile, the edges of the 128 x 64 tiles and of the 32 steps, rows that are not 16-byte aligned, a short block
@pytest.mark.parametrize("rows,cols,i1,i2", [(1, 132, 0, 128), (128, 192, 0, 128), (129, 320, 128, 256), (127, 193, 3, 128),
                                             (260, 300, 0, 33), (64, 8, 0, 4), (1000, 1411, 1280, 1408), (3, 129, 0, 128)])
def test_trailing_update(dev, rows, cols, i1, i2):
    g = torch.Generator().manual_seed(rows + cols)
    w, e, u = torch.randn(rows, cols, generator=g), torch.randn(rows, i2 - i1, generator=g), torch.randn(cols, cols, generator=g)
    got = w.to(dev)
    ops.gptq_trail(got, e.to(dev), u.to(dev), i1, i2)
    got = got.cpu()
    assert torch.equal(got[:, :i2], w[:, :i2]), "columns in front of the trailing part stay"
    prod = e.double() @ u[i1:i2, i2:].double()
    want = w[:, i2:].double() - prod
    # a sum of n products in any order is within n u sum|e||u| (u = 2^-24), the subtraction adds half a unit of its result
    bound = ((i2 - i1 + 1) * 2.0 ** -24) * (e.abs().double() @ u[i1:i2, i2:].abs().double()) + 2.0 ** -24 * want.abs() + 1e-30
    assert bool(((got[:, i2:].double() - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 1), (4, 100), (5, 4096), (7, 4097), (2, 9001)])
def test_column_order_and_back(dev, dtype, rows, cols):
    g = torch.Generator().manual_seed(cols)
    w = torch.randn(rows, cols, generator=g).to(dtype)
    perm, dead = torch.randperm(cols, generator=g), torch.rand(cols, generator=g) < 0.1
    ws = ops.gptq_order(w.to(dev), perm.to(dev), dead.to(dev))
    assert torch.equal(ws.cpu(), w.float().masked_fill(dead, 0)[:, perm])
    back = ops.gptq_order_back(ws, perm.to(dev), dtype)
    assert torch.equal(back.cpu(), w.masked_fill(dead, 0))
    values = torch.randn(rows, cols, generator=g)                  # rounded on the way back
    got = ops.gptq_order_back(values.to(dev), perm.to(dev), dtype).cpu()
    assert torch.equal(got, values[:, torch.argsort(perm)].to(dtype))
