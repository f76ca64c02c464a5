"""GPTQ inner-block kernel bit for bit against the oracle's restatement of
amct_pytorch/quantize_op/gptq_module.py:128-151, and the whole weight optimisation by tolerance (its
factorisations and GEMMs are library calls on both sides)."""
import pytest
import torch

from amct_amd import ops
from amct_amd.quantize_op import gptq
from oracle import gptq as og
from oracle import int_quant as iq
from util import assert_bits_equal

pytestmark = pytest.mark.gpu


def _hinv(count, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(count, 3 * count, generator=g)
    h = a @ a.t() / (3 * count) + 0.05 * torch.eye(count)
    c = torch.linalg.cholesky(torch.cholesky_inverse(torch.linalg.cholesky(h)), upper=True)
    return c.contiguous()


@pytest.mark.parametrize("kind,sym", [('int4', False), ('int4', True), ('int8', False), ('int8', True)])
@pytest.mark.parametrize("n,count,strategy", [(64, 128, 'channel'), (37, 40, 'channel'), (5, 1, 'channel'),
                                              (130, 128, 'group'), (16, 70, 'tensor'), (4100, 128, 'channel')])
def test_gptq_block_bit_exact(dev, kind, sym, n, count, strategy):
    g = torch.Generator().manual_seed(n * 7 + count)
    columns = count + 24                                            # the block sits inside a wider matrix
    w = (torch.randn(n, columns, generator=g) * 0.05).float()
    hinv_full = _hinv(columns, count)
    i1, i2 = 8, 8 + count
    bits = int(kind[3:])
    if strategy == 'group':
        G = 4
        wg = (torch.randn(n, G * 32, generator=g) * 0.05).float()
        s, z = iq.weight_scale_offset(wg, 'group', sym, kind, 32)
        s, z = s.reshape(n, G), (None if z is None else z.reshape(n, G))
        gidx = torch.randint(0, G, (count,), generator=g, dtype=torch.int32)
        scale_cols = [s[:, int(j)].unsqueeze(-1) for j in gidx]
        offset_cols = None if z is None else [z[:, int(j)].unsqueeze(-1) for j in gidx]
    else:
        s, z = iq.weight_scale_offset(w, strategy, sym, kind)
        gidx = torch.zeros(count, dtype=torch.int32)
        scale_cols = [s.reshape(-1, 1)] * count
        offset_cols = None if z is None else [z.reshape(-1, 1)] * count
    want_w = w.clone()
    _, want_e = og.block_loop(want_w[:, i1:i2], hinv_full[i1:i2, i1:i2], kind, scale_cols, offset_cols)
    dw = w.clone().to(dev)
    got_e = gptq.gptq_block(dw, i1, i2, hinv_full.to(dev), s.reshape(-1).contiguous().to(dev),
                            None if z is None else z.reshape(-1).to(torch.int32).contiguous().to(dev), gidx.to(dev),
                            -(1 << (bits - 1)), (1 << (bits - 1)) - 1)
    assert_bits_equal(got_e.cpu(), want_e, "err block")
    assert_bits_equal(dw.cpu(), want_w, "weight block (columns outside the block untouched)")


@pytest.mark.parametrize("n,count", [(70, 128), (33, 40)])
def test_gptq_block_full_matrix_hinv(dev, n, count):
    """A step only touches the columns at and behind its own (gptq_module.py:141): with an inverse-Hessian block
    that is NOT triangular the entries in front of the diagonal must be ignored, in both kernels (full 128-column
    blocks and shorter ones)."""
    g = torch.Generator().manual_seed(count)
    w = (torch.randn(n, count, generator=g) * 0.05).float()
    hinv = _hinv(count, 3) + 0.01 * torch.randn(count, count, generator=g)       # dense, diagonal still dominant
    s, z = iq.weight_scale_offset(w, 'channel', False, 'int4')
    gidx = torch.zeros(count, dtype=torch.int32)
    want_w = w.clone()
    _, want_e = og.block_loop(want_w, hinv, 'int4', [s.reshape(-1, 1)] * count, [z.reshape(-1, 1)] * count)
    dw = w.clone().to(dev)
    got_e = gptq.gptq_block(dw, 0, count, hinv.to(dev), s.reshape(-1).contiguous().to(dev),
                            z.reshape(-1).to(torch.int32).contiguous().to(dev), gidx.to(dev), -8, 7)
    assert_bits_equal(got_e.cpu(), want_e, "err block")
    assert_bits_equal(dw.cpu(), want_w, "weight block")


@pytest.mark.parametrize("strategy,group,sym", [('channel', None, True), ('group', 32, False)])
def test_gptq_whole_routine(dev, strategy, group, sym):
    """End to end.  The two sides factorise and multiply with different libraries, so a weight that sits next
    to a rounding boundary may land on the neighbouring code: nearly all entries agree closely, none differs
    by more than one quantisation step, and the layer output error of the two results is the same."""
    torch.manual_seed(3)
    n, k, t = 48, 256, 512
    w = (torch.randn(n, k) * 0.05).to(torch.bfloat16)
    x = torch.randn(t, k) * (1 + 3 * (torch.arange(k) % 17 == 0))
    x[:, 5] = 0                                                     # a dead input channel
    hess, ns = og.update_hessian(None, 0, x[:256], k)
    hess, ns = og.update_hessian(hess, ns, x[256:].reshape(2, 128, k), k)
    dh, dn = gptq.update_hessian(None, 0, x[:256].to(dev), k)
    dh, dn = gptq.update_hessian(dh, dn, x[256:].reshape(2, 128, k).to(dev), k)
    assert dn == ns
    torch.testing.assert_close(dh.cpu(), hess, rtol=1e-4, atol=1e-4)
    cfg = {'weights_cfg': {'quant_type': 'int4', 'symmetric': sym, 'strategy': strategy}}
    if group:
        cfg['weights_cfg']['group_size'] = group
    want, ws, wz = og.optimize_weight(w, hess, 'int4', strategy, sym, group)
    got, gs, gz = gptq.get_opt_weight_and_quant_factor(w.to(dev), hess.to(dev), cfg)
    assert got.dtype == w.dtype
    assert_bits_equal(gs.cpu().reshape(ws.shape), ws, "scale_w")
    diff = (got.cpu().float() - want.float()).abs()
    step = ws.reshape(n, -1).float().amax(dim=1, keepdim=True)
    assert (diff <= 1.01 * step + 1e-6).all()
    assert (diff <= 1e-3 * step).float().mean() > 0.97
    ref_err = ((x @ w.float().t()) - (x @ want.float().t())).pow(2).mean()
    got_err = ((x @ w.float().t()) - (x @ got.cpu().float().t())).pow(2).mean()
    assert abs(float(got_err) - float(ref_err)) <= 0.05 * float(ref_err)
    # and it is an improvement over plain rounding, which is the point of the algorithm
    plain = iq.fake_quant(w, 'int4', ws, wz, group)
    plain_err = ((x @ w.float().t()) - (x @ plain.float().t())).pow(2).mean()
    assert float(got_err) < float(plain_err)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,cols", [(256, 128), (1, 64), (63, 200), (65, 136), (1000, 520), (2048, 1024), (300, 4104), (77, 100), (130, 1099)])
def test_hessian_update_kernel(dev, dtype, tokens, cols):
    """H <- beta H + alpha X^T X (gptq_module.py:176-181) on the matrix pipe.  Small integers make every product
    and sum exact in fp32, so the first call (beta = 0, H full of NaN beforehand: it must not be read) and a second,
    accumulating call are compared bit for bit with an integer matmul; random activations are compared with the fp64
    product at the fp32 rounding of a sum of that many terms.  Ragged tokens and columns; H comes out exactly symmetric."""
    from amct_amd import ops
    g = torch.Generator().manual_seed(tokens * 31 + cols)
    xi = torch.randint(-4, 5, (tokens, cols), generator=g)
    h = torch.full((cols, cols), float('nan'), dtype=torch.float32, device=dev)
    ops.hessian_update(h, xi.to(dtype).to(dev), 0.0, 1.0)
    want = (xi.double().t() @ xi.double())
    assert_bits_equal(h, want.float() + 0.0, "first call, integers")     # (+ 0.0: a sum that starts at +0 never ends at -0)
    xj = torch.randint(-4, 5, (max(tokens // 2, 1), cols), generator=g)
    ops.hessian_update(h, xj.to(dtype).to(dev), 0.5, 2.0)            # powers of two: still exact
    want = 0.5 * want + 2.0 * (xj.double().t() @ xj.double())
    assert_bits_equal(h, want.float() + 0.0, "second call, integers")
    x = torch.randn(tokens, cols, generator=g).to(dtype)
    h0 = torch.randn(cols, cols, generator=g)
    h0 = (h0 + h0.t()).contiguous()
    hd = h0.clone().to(dev)
    beta, alpha = 0.75, 2.0 / (tokens + 7)
    ops.hessian_update(hd, x.to(dev), beta, alpha)
    ref = beta * h0.double() + alpha * (x.double().t() @ x.double())
    mag = beta * h0.double().abs() + alpha * (x.double().abs().t() @ x.double().abs())
    err = (hd.cpu().double() - ref).abs()
    assert (err <= 2.0 ** -20 * mag + 1e-30).all(), float((err / (mag + 1e-30)).max())
    assert torch.equal(hd, hd.t()), "symmetry"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,cols", [(64, 64), (128, 72), (191, 2432), (1, 2433), (65, 2440), (257, 3968), (130, 3969), (64, 4224), (200, 4225), (449, 4300)])
def test_hessian_tiles(dev, dtype, tokens, cols):
    """Both sides of the lines between the tile widths, whole and partial last steps and tiles, X and H that start off a
    16-byte boundary: sums of small integers are exact, so every element is compared bit for bit; nothing is written behind
    the matrix."""
    g = torch.Generator().manual_seed(tokens + cols)
    for off in (0, 1):
        x = torch.empty(tokens * cols + 8, dtype=dtype, device=dev)[off:off + tokens * cols].view(tokens, cols)
        x.copy_(torch.randint(-4, 5, (tokens, cols), generator=g))
        buf = torch.full((cols * cols + 200,), 7.0, device=dev)
        h = buf[off:off + cols * cols].view(cols, cols)
        h.fill_(float('nan'))
        prod = x.double().t() @ x.double()
        ops.hessian_update(h, x, 0.0, 1.0)
        assert torch.equal(h.double(), prod)
        ops.hessian_update(h, x, 0.5, 2.0)
        assert torch.equal(h.double(), 2.5 * prod)
        assert bool((buf[:off] == 7).all()) and bool((buf[off + cols * cols:] == 7).all())


def test_update_hessian_on_16_bit_activations(dev):
    """quantize_op.gptq.update_hessian with bf16 activations on the device takes the kernel; against the oracle's
    restatement of the reference (fp32 product of the scaled activations) within the rounding of the two orders of
    operations."""
    torch.manual_seed(5)
    k = 384
    x = (torch.randn(640, k) * (1 + 3 * (torch.arange(k) % 17 == 0))).to(torch.bfloat16)
    hess, ns = og.update_hessian(None, 0, x[:256], k)
    hess, ns = og.update_hessian(hess, ns, x[256:].reshape(3, 128, k), k)
    dh, dn = gptq.update_hessian(None, 0, x[:256].to(dev), k)
    dh, dn = gptq.update_hessian(dh, dn, x[256:].reshape(3, 128, k).to(dev), k)
    assert dn == ns and dh.dtype == torch.float32
    torch.testing.assert_close(dh.cpu(), hess, rtol=1e-4, atol=1e-4)
    # both are fp32 sums in different orders; against the same recurrence in fp64 the kernel is the closer one or as close
    xd = x.double()
    exact = (2 / 1) * (xd[:256].t() @ xd[:256]) * (1 / 1)            # first call: nsamples 0 -> 1
    exact = exact * (1 / 4) + (2 / 4) * (xd[256:].t() @ xd[256:])    # second call: batch of 3, nsamples 1 -> 4
    mine, theirs = (dh.cpu().double() - exact).abs().max(), (hess.double() - exact).abs().max()
    assert float(mine) <= 1.5 * float(theirs) + 1e-6, (float(mine), float(theirs))


@pytest.mark.parametrize("sym", [False, True])
@pytest.mark.parametrize("n", [1, 4, 17, 63, 300, 8192, 8193])
@pytest.mark.parametrize("special", ['none', 'tiny weights', 'huge weights', 'inf weight', 'tiny scale', 'tiny diagonal'])
def test_gptq_full_block_is_the_general_kernel(dev, sym, n, special):
    """Full blocks divide by reciprocals while everything stays in the range where that gives the quotient's bits, and
    by the division itself in the waves that leave it: the bits of the general kernel, which an odd row stride selects."""
    g = torch.Generator().manual_seed(n)
    count = 128
    w = (torch.randn(n, count, generator=g) * 0.05).float()
    s, z = iq.weight_scale_offset(w, 'channel', sym, 'int4')
    s, z = s.reshape(n, 1).repeat(1, 2), None if z is None else z.reshape(n, 1).repeat(1, 2)
    s[:, 1] *= 1.25
    hinv = _hinv(count, 5)
    row = n // 2
    w[row, 3] = -0.0
    if special == 'tiny weights':
        w[row, 40:44] = torch.tensor([1e-38, -1e-42, 1e-25, -1e-20])
        hinv = hinv * torch.eye(count)                              # nothing is added to them on the way
    elif special == 'huge weights':
        w[row, 7], w[row, 100] = 1e30, -3e38
    elif special == 'inf weight':
        w[row, 64] = float('inf')
    elif special == 'tiny scale':
        s[row, 1] = 1e-30
    elif special == 'tiny diagonal':
        hinv[17, 17] = 1e-25
    gidx = torch.randint(0, 2, (count,), generator=g, dtype=torch.int32)
    factors = (s.contiguous().to(dev), None if z is None else z.to(torch.int32).contiguous().to(dev), gidx.to(dev))
    padded = torch.full((n, count + 1), 7.0, device=dev)
    padded[:, :count] = w.to(dev)
    want_e = gptq.gptq_block(padded, 0, count, hinv.to(dev), *factors, -8, 7)
    got = w.to(dev)
    got_e = gptq.gptq_block(got, 0, count, hinv.to(dev), *factors, -8, 7)
    assert_bits_equal(got_e.nan_to_num(1.5).cpu(), want_e.nan_to_num(1.5).cpu(), "err block")
    assert torch.equal(got_e.isnan(), want_e.isnan())
    assert_bits_equal(got.nan_to_num(1.5).cpu(), padded[:, :count].contiguous().nan_to_num(1.5).cpu(), "weight block")
    assert torch.equal(got.isnan(), padded[:, :count].isnan())


@pytest.mark.parametrize("cols", [8, 130, 300])
@pytest.mark.parametrize("where", [None, 'first', 'last', 'overflow', 'old'])
def test_hessian_update_reports_what_is_not_finite(dev, cols, where):
    x = torch.ones(5, cols, dtype=torch.bfloat16, device=dev)
    h = torch.ones(cols, cols, device=dev)
    if where == 'first':
        x[0, 0] = float('nan')
    elif where == 'last':
        x[4, cols - 1] = float('inf')
    elif where == 'overflow':
        x[2, cols // 2] = 3e38
    elif where == 'old':
        h[cols - 1, 0] = h[0, cols - 1] = float('-inf')
    bad = torch.full((1,), 7, dtype=torch.int32, device=dev)
    for _ in range(2):
        ops.hessian_update(h, x, 0.5, 0.5, bad)
        assert int(bad) == int(where is not None) == int(not bool(torch.isfinite(h).all()))


@pytest.mark.parametrize("columns", [64, 300])
@pytest.mark.parametrize("sym", [False, True])
def test_gptq_whole_routine_raises_what_the_kernels_report(dev, columns, sym):
    """The flags of the factors and of the factorisation are read behind everything that is enqueued (several blocks of
    columns at 300): each raises the error of its own, the factors' first, and a valid layer raises none."""
    g = torch.Generator().manual_seed(columns)
    w = torch.randn(24, columns, generator=g) * 0.05
    x = torch.randn(3 * columns, columns, generator=g)
    hess = (x.t() @ x).div(x.shape[0]).to(dev)
    cfg = {'weights_cfg': {'quant_type': 'int4', 'symmetric': sym, 'strategy': 'channel'}}
    spoilt = []
    for value in (float('inf'), float('nan')):
        spoilt.append(w.clone())
        spoilt[-1][7, columns - 1] = value
    indefinite = hess.clone()
    indefinite[3, columns - 2] = indefinite[columns - 2, 3] = 50.
    with_nan = hess.clone()
    with_nan[columns // 2, columns // 2] = float('nan')
    for _ in range(2):
        for bad in spoilt:
            for h in (hess, indefinite):
                with pytest.raises(RuntimeError, match="Param scale has invalid value inf, nan or zeros!"):
                    gptq.get_opt_weight_and_quant_factor(bad.to(dev), h, cfg)
        for h in (indefinite, with_nan):
            with pytest.raises(torch.linalg.LinAlgError, match="not positive-definite"):
                gptq.get_opt_weight_and_quant_factor(w.to(dev), h, cfg)
        got = gptq.get_opt_weight_and_quant_factor(w.to(dev), hess, cfg)[0]
        assert bool(torch.isfinite(got).all())


def _parts(x, width):
    """x fp32 [N, K] as three bf16 parts [N, 3, width], the leading K columns of each."""
    out = torch.empty(x.shape[0], 3, width, dtype=torch.bfloat16, device=x.device)
    rest = x.clone()
    for k in range(3):
        out[:, k, :x.shape[1]] = rest.bfloat16()
        rest = rest - out[:, k, :x.shape[1]].float()
    return out[:, :, :x.shape[1]]


@pytest.mark.parametrize("n,columns,i1,i2,end", [(1, 65, 0, 32, 65), (63, 200, 32, 64, 136), (64, 192, 0, 128, 192), (65, 321, 96, 256, 321),
                                                 (300, 1000, 0, 512, 1000), (1100, 777, 64, 608, 777), (130, 900, 160, 192, 193)])
@pytest.mark.parametrize("spread", [0.0, 2.0])
def test_gptq_trail_from_parts(dev, n, columns, i1, i2, end, spread):
    """The update from three bf16 parts against the fp64 product.  Left out of a product: below 2^-25 of it.  A sum of 128
    steps takes 6 * 128 / 32 additions of a wave's partial sums; the additions inside an instruction are taken to round
    as often again; two units each bound what the hardware rounds by.  Every 128 steps one more rounding as W is updated.  The
    products alone (W zero: its rounding every 128 steps is the reference's) are on the whole no further off than those of
    the fp32 kernel taken 128 steps at a time (of values of one size: with a wide spread a handful of elements decides)."""
    g = torch.Generator().manual_seed(n + columns)
    err = (torch.randn(n, i2 - i1, generator=g) * torch.exp(spread * torch.randn(n, i2 - i1, generator=g)) * 0.01).to(dev)
    err[torch.rand(n, i2 - i1, generator=g).to(dev) < 0.1] = 0.
    u = torch.triu(torch.randn(columns, columns, generator=g) * torch.exp(spread * torch.randn(columns, columns, generator=g))).to(dev)
    w = torch.randn(n, columns, generator=g).to(dev)
    wide = torch.zeros(1, dtype=torch.int32, device=dev)
    u_parts = ops.gptq_split(u, wide)
    rows, cols = torch.triu_indices(columns, columns, device=dev)
    assert torch.equal(u_parts.double().sum(1)[rows, cols], u.double()[rows, cols]) and int(wide) == 0
    err_parts = _parts(err, (i2 - i1 + 63) // 32 * 32)
    ref = w.double()
    ref[:, i2:end] -= err.double() @ u[i1:i2, i2:end].double()
    mag = err.double().abs() @ u[i1:i2, i2:end].double().abs()
    for flag in (0, 1):                                   # the parts, the fp32 values themselves
        got = w.clone()
        ops.gptq_trail_parts(got, err, u, err_parts, u_parts, torch.full_like(wide, flag), i1, i2, end)
        assert torch.equal(got[:, :i2], w[:, :i2]) and torch.equal(got[:, end:], w[:, end:])
        off = (got.double() - ref).abs()[:, i2:end]
        sums = -(-(i2 - i1) // 128)
        bound = (2 * 2 * 24 + 2) * 2.0 ** -24 * mag + sums * 2.0 ** -24 * (w[:, i2:end].double().abs() + mag)
        if flag:
            bound = bound + 128 * 2.0 ** -24 * mag        # one rounding a step instead
        assert bool((off <= bound).all()), float((off / bound).max())
    if spread:
        return
    product = ref[:, i2:end] - w[:, i2:end].double()
    off = []
    for flag in (0, 1):
        got = torch.zeros_like(w)
        ops.gptq_trail_parts(got, err, u, err_parts, u_parts, torch.full_like(wide, flag), i1, i2, end)
        off.append(float((got[:, i2:end].double() - product).norm()))
    assert off[0] <= off[1], off


@pytest.mark.parametrize("value", [float('inf'), float('nan'), 2.0 ** 60, -2.0 ** 127, 2.0 ** -101, 2.0 ** -140])
def test_gptq_parts_say_what_they_do_not_hold(dev, value):
    u = torch.triu(torch.ones(130, 130)).to(dev)
    for at in ((0, 0), (3, 129), (129, 129)):
        wide = torch.zeros(1, dtype=torch.int32, device=dev)
        spoilt = u.clone()
        spoilt[at] = value
        ops.gptq_split(spoilt, wide)
        assert int(wide) == 1
    for kept in (0.0, -0.0, 2.0 ** -100, -(2.0 ** 60) * (1 - 2.0 ** -24)):
        wide.zero_()
        kind = u.clone()
        kind[5, 77] = kept
        ops.gptq_split(kind, wide)
        assert int(wide) == 0


@pytest.mark.parametrize("columns,block_size", [(1025, 128), (1300, 96), (1100, 640)])
def test_gptq_layer_by_spans(dev, monkeypatch, columns, block_size):
    """Spans of columns updated from parts against one fp32 update per block.  The two differ by roundings, which move a code
    where one sits on a rounding boundary, and with it codes behind it in its row: few rows, if any, and the layer's error
    on its inputs is the same to a thousandth."""
    g = torch.Generator().manual_seed(columns)
    w = (torch.randn(90, columns, generator=g) * 0.05).to(dev)
    x = torch.randn(2 * columns, columns, generator=g).to(dev)
    x[:, ::97] *= 5
    hess = (x.t() @ x).div(x.shape[0])
    cfg = {'weights_cfg': {'quant_type': 'int4', 'symmetric': False, 'strategy': 'channel'}}
    if block_size > 128:
        with pytest.raises(RuntimeError):
            gptq.get_opt_weight_and_quant_factor(w, hess, cfg, block_size=block_size)
        return
    spans = gptq.get_opt_weight_and_quant_factor(w, hess, cfg, block_size=block_size)
    monkeypatch.setattr(gptq, '_PARTS_COLUMNS', (1, 0))
    blocks = gptq.get_opt_weight_and_quant_factor(w, hess, cfg, block_size=block_size)
    assert torch.equal(spans[1], blocks[1]) and torch.equal(spans[2], blocks[2])
    moved = ((spans[0] - blocks[0]).abs() > 0.5 * spans[1].reshape(-1, 1)).any(1)
    assert int(moved.sum()) <= 5
    # (what the column loop leaves is w - err * hinv[i][i], the code's value up to three roundings of numbers below 32 steps)
    assert bool(((spans[0] - blocks[0]).abs() <= 2 * 3 * 32 * 2.0 ** -24 * spans[1].reshape(-1, 1))[~moved].all())
    off = [float((x @ (w - o[0]).t()).double().pow(2).sum()) for o in (spans, blocks)]
    assert abs(off[0] / off[1] - 1) <= 1e-3


@pytest.mark.parametrize("n,count", [(1, 128), (70, 128), (9000, 128), (33, 32), (64, 100)])
def test_gptq_block_gives_its_errors_in_parts(dev, n, count):
    g = torch.Generator().manual_seed(n + count)
    w = torch.randn(n, count, generator=g).to(dev)
    hinv = _hinv(count, count).to(dev)
    scale = torch.full((n,), 0.1, device=dev)
    gidx = torch.zeros(count, dtype=torch.int32, device=dev)
    want_w = w.clone()
    want = gptq.gptq_block(want_w, 0, count, hinv, scale, None, gidx, -8, 7)
    errors = torch.zeros(n, count + 28, device=dev)
    parts = torch.zeros(n, 3, count + 28, dtype=torch.bfloat16, device=dev)
    wide = torch.zeros(1, dtype=torch.int32, device=dev)
    got = gptq.gptq_block(w, 0, count, hinv, scale, None, gidx, -8, 7, errors[:, :count], parts[:, :, :count], wide)
    assert torch.equal(got, want) and torch.equal(w, want_w) and int(wide) == 0
    assert torch.equal(parts[:, :, :count].double().sum(1), want.double())
    assert not bool(errors[:, count:].any()) and not bool(parts[:, :, count:].any())
    w = want_w.clone()
    w[n // 2, count // 3] = float('inf')
    gptq.gptq_block(w, 0, count, hinv, scale, None, gidx, -8, 7, errors[:, :count], parts[:, :, :count], wide)
    assert int(wide) == 1


@pytest.mark.parametrize("columns", [3, 64, 66, 1020, 1027, 2052, 4100])
def test_gptq_factor_of_a_matrix_off_16_bytes(dev, columns):
    """Rows fetched 16 bytes at a time (columns a multiple of 4, an aligned matrix) and word by word hold the same values: the same
    factor bit for bit, for one piece of a lane's loads and for more."""
    x = torch.randn(2 * columns, columns, device=dev, generator=torch.Generator(dev).manual_seed(columns))
    h = x.t() @ x / (2 * columns)
    h = (h + h.t()) / 2
    perm = torch.randperm(columns, device=dev)
    damp = torch.tensor(0.01, device=dev)
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    shifted = torch.empty(columns * columns + 1, device=dev)[1:].view(columns, columns)
    shifted.copy_(h)
    assert torch.equal(ops.gptq_factor(h, perm, damp, bad), ops.gptq_factor(shifted, perm, damp, bad)) and int(bad) == 0
