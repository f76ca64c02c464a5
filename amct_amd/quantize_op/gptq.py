"""Host-side mirror of the weight optimisation of amct_pytorch/quantize_op/gptq_module.py (:91-155, :161-186)
with the tensors resident on the device.  The column loop of each block is one kernel launch (amct_gptq_block), the
update of the columns behind it another (amct_gptq_trail, of wide layers amct_gptq_trail_parts), the factorisations one call
(amct_gptq_factor)."""
import math

import torch

from .. import _lib, ops
from .utils import check_scale_offset, get_weight_min_max_by_granularity


@torch.no_grad()
def update_hessian(hessian, nsamples, input_data, columns):
    """:161-186.  Returns (hessian, nsamples); the matrix stays on the device instead of moving to the host.
    For bf16 / fp16 activations on the device the update runs in place: the returned tensor IS the `hessian` passed in
    (the reference and the fp32 branch below build a new tensor per call) -- pass a clone to keep the earlier value.
    That branch applies 2 / n to the fp32 sum of exact products instead of scaling every element by sqrt(2 / n) first,
    so it matches the reference to fp32 rounding, not bit for bit."""
    if len(input_data.shape) == 2:
        input_data = input_data.unsqueeze(0)
    batch_size = input_data.shape[0]
    rows = input_data.reshape((-1, input_data.shape[-1]))
    if rows.is_cuda and rows.dtype in (torch.bfloat16, torch.float16):
        # the matrix-pipe kernel: one pass over the lower triangle of H, the product of the 16-bit values exact in fp32
        if hessian is None:
            hessian = torch.empty((columns, columns), dtype=torch.float32, device=rows.device)
            beta = 0.0
        else:
            beta = nsamples / (nsamples + batch_size)
        nsamples += batch_size
        hessian, bad = ops.with_host_flag(
            rows, lambda flag: ops.hessian_update(hessian, rows, beta, 2 / nsamples, flag=flag))
        finite = not bad
    else:
        # fp32 activations keep the fp32 product
        x = rows.t()
        if hessian is None:
            hessian = torch.zeros((columns, columns), device=x.device)
        hessian = hessian * (nsamples / (nsamples + batch_size))
        nsamples += batch_size
        x = math.sqrt(2 / nsamples) * x.float()
        hessian = hessian + x.matmul(x.t())
        finite = bool(torch.isfinite(hessian).all())
    if not finite:
        raise RuntimeError("hessian matrix has invalid value, inf or nan.")
    return hessian, nsamples


# Columns whose errors are kept for one update of everything behind them; inside, a block's update reaches the end of these
# columns only.  The weight is read and written once per 512 columns instead of once per 128, and the products of one update
# are enough to keep the matrix pipe busy.
_SPAN = 512
# From how many columns on, and to how many (the parts of the factor are 6 bytes an element: 1.6 GB).  W[1024,1024]: 0.53 ms both
# ways, of 512 columns 0.33 with spans and 0.31 without (the launches count there), W[1024,5120] 3.30 and 3.42, W[4096,4096]
# 2.66 and 2.98, W[14336,4096] 4.45 and 5.21.
_PARTS_COLUMNS = (1025, 16384)


def gptq_block(weight_sorted, i1, i2, hinv, scale_w, offset_w, gidx, qmin, qmax, err=None, parts=None, wide=None):
    """The column loop of block [i1, i2) in place on weight_sorted [N, columns] fp32; returns err_block, written to err, where
    given: the columns [N, i2 - i1] of a wider matrix.  parts: the same columns of [N, 3, ...] bf16, err_block as the sum of
    three; wide (int32, one element) becomes 1 where they do not hold it."""
    dev = ops._dev(weight_sorted, hinv, scale_w, offset_w, gidx)
    n, columns = weight_sorted.shape
    count = i2 - i1
    if err is None:
        err = torch.empty(n, count, dtype=torch.float32, device=dev)
    if scale_w.numel() == 1:
        stride = 0
    else:
        stride = scale_w.numel() // n
    w_ptr = weight_sorted.data_ptr() + i1 * 4
    h_ptr = hinv.data_ptr() + (i1 * hinv.shape[1] + i1) * 4
    with torch.cuda.device(dev):
        _lib.check(_lib.load().amct_gptq_block_parts(
            w_ptr, columns, err.data_ptr(), err.stride(0), h_ptr, hinv.shape[1], scale_w.data_ptr(),
            None if offset_w is None else offset_w.data_ptr(), stride, gidx.data_ptr(), n, count, qmin, qmax,
            None if parts is None else parts.data_ptr(), 0 if parts is None else parts.stride(1),
            None if wide is None else wide.data_ptr(), torch.cuda.current_stream(dev).cuda_stream))
    return err


def _read_later(flag):
    """(host copy of a device flag, event behind the copy): read the copy after event.synchronize(), which waits for the
    work up to here and not for what is enqueued behind it.  The copy runs on the current stream of the flag's device, which
    need not be the current device: the event is recorded there."""
    host = torch.empty(flag.shape, dtype=flag.dtype, pin_memory=True)
    host.copy_(flag, non_blocking=True)
    event = torch.cuda.Event()
    event.record(torch.cuda.current_stream(flag.device))
    return host, event


def _by_spans(ws, hinv, scale_w, offset_w, gidx, qmin, qmax, block_size, wide):
    """The blocks of ws [N, columns] with their updates made by spans of columns, from the parts of the errors and of hinv."""
    rows, columns = ws.shape
    span = max(1, _SPAN // block_size) * block_size
    width = min(span, -(-columns // 32) * 32)
    hinv_parts = ops.gptq_split(hinv, wide)
    errors = torch.empty(rows, width, dtype=torch.float32, device=ws.device)
    parts = torch.empty(rows, 3, width, dtype=torch.bfloat16, device=ws.device)
    for s1 in range(0, columns, span):
        s2 = min(s1 + span, columns)
        for i1 in range(s1, s2, block_size):
            i2 = min(i1 + block_size, s2)
            at = slice(i1 - s1, i2 - s1)
            gptq_block(ws, i1, i2, hinv, scale_w, offset_w, gidx[i1:i2].contiguous(), qmin, qmax, errors[:, at], parts[:, :, at], wide)
            if i2 < s2:
                ops.gptq_trail_parts(ws, errors[:, at], hinv, parts[:, :, at], hinv_parts, wide, i1, i2, s2)
        if s2 < columns:
            ops.gptq_trail_parts(ws, errors[:, :s2 - s1], hinv, parts[:, :, :s2 - s1], hinv_parts, wide, s1, s2, columns)


@torch.no_grad()
def get_opt_weight_and_quant_factor(weight, hessian, quant_config, block_size=128, perc_damp=0.01):
    """:91-155.  weight [N, K] (any float dtype), hessian [K, K] fp32 on the same device.  Returns
    (optimised weight in the weight's dtype, scale_w, offset_w)."""
    cfg = quant_config.get('weights_cfg')
    group_size = cfg.get('group_size')
    wts_type = cfg.get('quant_type')
    bits = int(wts_type.replace('int', ''))
    columns = weight.shape[1]
    out_dtype = weight.dtype
    if out_dtype not in (torch.float32, torch.float16, torch.bfloat16):
        weight = weight.float()
    hessian = hessian.float()
    diag = torch.diag(hessian)
    dead = diag == 0
    diag = torch.where(dead, torch.ones_like(diag), diag)
    perm = torch.argsort(diag, descending=True)
    # the extrema of the weight with its dead columns at zero, in fp32 like the weight that the reference works on
    weight_min, weight_max = get_weight_min_max_by_granularity(weight.masked_fill(dead, 0), quant_config)
    # flags that the kernels raise: a factor not finite, a pivot not positive (read when everything is enqueued), a value that
    # three bf16 parts do not hold (read by the updates)
    bad = torch.zeros(3, dtype=torch.int32, device=weight.device)
    scale_w, offset_w = ops.scale_offset(weight_max.float(), weight_min.float(), bits, bool(cfg.get('symmetric')), bad=bad[:1])
    ws = ops.gptq_order(weight, perm, dead)
    # cholesky(cholesky_inverse(cholesky(hs)), upper=True) of the permuted, damped Hessian, as one factorisation
    hinv = ops.gptq_factor(hessian, perm, perc_damp * torch.mean(diag), bad[1:2])
    flags, factored = _read_later(bad)
    sc = scale_w.reshape(-1).float().contiguous()
    zc = None if offset_w is None else offset_w.reshape(-1).to(torch.int32).contiguous()
    if group_size:
        gidx_all = (perm // group_size).to(torch.int32)
    else:
        gidx_all = torch.zeros(columns, dtype=torch.int32, device=weight.device)
    qmin, qmax = -(1 << (bits - 1)), (1 << (bits - 1)) - 1
    if block_size % 32 == 0 and _PARTS_COLUMNS[0] <= columns <= _PARTS_COLUMNS[1]:
        _by_spans(ws, hinv, sc, zc, gidx_all, qmin, qmax, block_size, bad[2:])
    else:
        for i1 in range(0, columns, block_size):
            i2 = min(i1 + block_size, columns)
            err_block = gptq_block(ws, i1, i2, hinv, sc, zc, gidx_all[i1:i2].contiguous(), qmin, qmax)
            if i2 < columns:
                ops.gptq_trail(ws, err_block, hinv, i1, i2)
    result = ops.gptq_order_back(ws, perm, weight.dtype).to(out_dtype)
    factored.synchronize()                          # of the copy only: long done when the last block is enqueued
    if int(flags[0]):
        check_scale_offset(scale_w, None)
        raise RuntimeError("Param offset has invalid value inf or nan!")
    if int(flags[1]):
        raise torch.linalg.LinAlgError("linalg.cholesky: the factorization could not be completed because the input is "
                                       "not positive-definite.")
    return result, scale_w, offset_w
