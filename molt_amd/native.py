"""Whole directions of the autograd nodes as one library call each
(``molt_linear_*``, ``molt_gated_mlp_*``, ``molt_stacked_*`` of
include/molt_amd.h): the same kernels in the same order as the separate ops of
``molt_amd.ops``, issued from native code out of one workspace, so the results
are theirs bit for bit.

Each function returns None for a call it does not take: under torch.compile or
with event probes on, with tensors that are not plain, contiguous, of the
kernels' dtypes and on one device, or of shapes that do not match. The caller
then runs the separate ops, which convert what can be converted and raise for
the rest.
"""
from __future__ import annotations

import ctypes as C
from typing import Any, Optional

import torch
from torch import Tensor

from . import _lib, ops
from .nf4 import _rows_cols, nibble_order, resolved_nf4_scales

_PLAIN = (Tensor, torch.nn.Parameter)
_BF16, _F32, _U8 = torch.bfloat16, torch.float32, torch.uint8
MAX_RANK = 128


def _off() -> bool:
    return bool(ops._probes) or torch.compiler.is_compiling()


def _is(t: Tensor, dtype: torch.dtype, dev: int) -> bool:
    return type(t) in _PLAIN and t.dtype is dtype and t.get_device() == dev and t.is_contiguous()


def _rows(t: Tensor, dev: int, m: int, n: int) -> bool:
    return _is(t, _BF16, dev) and t.shape == (m, n)


def _adapter(t: Tensor, dev: int, rows: int, cols: int) -> bool:
    return _is(t, _F32, dev) and t.shape == (rows, cols)


def _weight(packed: Tensor, qs: Any, dev: int) -> Optional[_lib.NF4Weight]:
    """The weight's descriptor, or None. The caller keeps packed and qs alive
    over the launch; the resolved scales are cached on qs."""
    n, k = _rows_cols(qs.shape)
    block = int(qs.blocksize)
    scales, code = resolved_nf4_scales(qs), qs.code
    if not (_is(packed, _U8, dev) and packed.numel() * 2 >= n * k and _is(scales, _F32, dev) and block > 0
            and scales.numel() * block >= n * k and _is(code, _F32, dev) and code.numel() >= 16):
        return None
    return ops._weight(packed, scales, code, n, k, block, nibble_order(qs))


def _empty(dev: torch.device, dtype: torch.dtype, *shape: int) -> Tensor:
    return torch.empty(shape, device=dev, dtype=dtype)


def _packed_b(dev: torch.device, rows: int, r: int) -> Tensor:
    return _empty(dev, _U8, ops._workspace("molt_lora_packed_bytes", rows, r))


# ------------------------------------------------------------ one projection
def linear_forward(x: Tensor, packed: Tensor, a: Tensor, b: Tensor, qs: Any, s: float, grad: bool, keep: bool):
    """(Y, T, packed B or None, deq(W)^T or None) of a scheduled projection."""
    if _off() or x.dim() != 2 or not x.is_cuda:
        return None
    n, k = _rows_cols(qs.shape)
    dev, m, r = x.get_device(), x.shape[0], a.shape[0]
    if not (m > 0 and 0 < r <= MAX_RANK and _rows(x, dev, m, k) and _adapter(a, dev, r, k) and _adapter(b, dev, n, r)):
        return None
    w = _weight(packed, qs, dev)
    if w is None:
        return None
    d = x.device
    y, t = _empty(d, _BF16, m, n), _empty(d, _BF16, m, r)
    bp = _packed_b(d, n, r) if grad else None
    wt = _empty(d, _BF16, k, n) if keep and ops._keeps_wt(m, n, k, 1) else None
    written = C.c_int32(0)
    size = ops._workspace("molt_linear_forward_workspace", m, n, k, r)
    ws = _empty(d, _U8, size)
    ops._call("molt_linear_forward", x.data_ptr(), m, w, a.data_ptr(), b.data_ptr(), r, s, ops._ptr(bp),
              t.data_ptr(), y.data_ptr(), ops._ptr(wt), C.byref(written) if wt is not None else None, ws.data_ptr(),
              size, ops._stream(d))
    return y, t, bp, wt if written.value else None


def linear_backward(dy: Tensor, x: Tensor, t: Tensor, packed: Tensor, a: Tensor, bp: Optional[Tensor], qs: Any, s: float,
                    wt: Optional[Tensor]):
    """(dX, dA, dB) of a scheduled projection."""
    if bp is None or _off() or not dy.is_cuda:
        return None
    n, k = _rows_cols(qs.shape)
    dev, m, r = dy.get_device(), x.shape[0], a.shape[0]
    if not (m > 0 and _rows(dy, dev, m, n) and _rows(x, dev, m, k) and _rows(t, dev, m, r)
            and _adapter(a, dev, r, k) and bp.get_device() == dev and (wt is None or _rows(wt, dev, k, n))):
        return None
    w = _weight(packed, qs, dev)
    if w is None:
        return None
    d = dy.device
    dx, da, db = _empty(d, _BF16, m, k), _empty(d, _F32, r, k), _empty(d, _F32, n, r)
    size = ops._workspace("molt_linear_backward_workspace", m, n, k, r, int(wt is not None))
    ws = _empty(d, _U8, size)
    ops._call("molt_linear_backward", dy.data_ptr(), x.data_ptr(), t.data_ptr(), m, w, a.data_ptr(), bp.data_ptr(), r,
              s, ops._ptr(wt), dx.data_ptr(), da.data_ptr(), db.data_ptr(), ws.data_ptr(), size, ops._stream(d))
    return dx, da, db


# ------------------------------------------------------------- the gated MLP
def _mlp_weights(gate, up, down, qs, dev: int):
    if any(int(q.blocksize) != 64 for q in qs) or nibble_order(qs[0]) != nibble_order(qs[1]):
        return None
    ws = [_weight(p, q, dev) for p, q in zip((gate, up, down), qs)]
    if any(w is None for w in ws):
        return None
    if ws[1].code != ws[0].code:      # the paired GEMMs read one code table: the gate's, as the separate ops do
        ws[1] = ops._weight(up, resolved_nf4_scales(qs[1]), qs[0].code, ws[1].rows, ws[1].cols, 64, ws[1].nibble_order)
    return ws


def mlp_forward(x: Tensor, packed: tuple, adapters: tuple, qs: tuple, scaling: tuple, grad: bool, keep: bool):
    """(Y, gate, up, h, T_gu, T_d, (B_d, B_g, B_u packed) or None) of the gated
    MLP; ``adapters`` is (A_g, B_g, A_u, B_u, A_d, B_d). A batch whose GEMMs
    would hand their weights to the backward takes the separate ops."""
    if _off() or x.dim() != 2 or not x.is_cuda:
        return None
    i, h = _rows_cols(qs[0].shape)
    dev, m = x.get_device(), x.shape[0]
    ag, bg, au, bu, ad, bd = adapters
    r = ag.shape[0]
    if not (m > 0 and 0 < 2 * r <= MAX_RANK and _rows(x, dev, m, h)
            and _rows_cols(qs[1].shape) == (i, h) and _rows_cols(qs[2].shape) == (h, i)
            and _adapter(ag, dev, r, h) and _adapter(au, dev, r, h) and _adapter(ad, dev, r, i)
            and _adapter(bg, dev, i, r) and _adapter(bu, dev, i, r) and _adapter(bd, dev, h, r)):
        return None
    if keep and (ops._keeps_wt(m, i, h, 2) or ops._keeps_wt(m, h, i, 1)):
        return None
    ws = _mlp_weights(*packed, qs, dev)
    if ws is None:
        return None
    d = x.device
    gate, up, hid = (_empty(d, _BF16, m, i) for _ in range(3))
    y, t_gu, t_d = _empty(d, _BF16, m, h), _empty(d, _BF16, m, 2 * r), _empty(d, _BF16, m, r)
    bps = (_packed_b(d, h, r), _packed_b(d, i, r), _packed_b(d, i, r)) if grad else None
    size = ops._workspace("molt_gated_mlp_forward_workspace", m, h, i, r)
    buf = _empty(d, _U8, size)
    ops._call("molt_gated_mlp_forward", x.data_ptr(), m, *ws, ag.data_ptr(), bg.data_ptr(), au.data_ptr(),
              bu.data_ptr(), ad.data_ptr(), bd.data_ptr(), r, *scaling,
              *((p.data_ptr() for p in bps) if grad else (None, None, None)), t_gu.data_ptr(), t_d.data_ptr(),
              gate.data_ptr(), up.data_ptr(), hid.data_ptr(), y.data_ptr(), buf.data_ptr(), size, ops._stream(d))
    return y, gate, up, hid, t_gu, t_d, bps


def mlp_backward(dy: Tensor, x: Tensor, gate: Tensor, up: Tensor, hid: Optional[Tensor], t_gu: Tensor, t_d: Tensor,
                 packed: tuple, adapters: tuple, qs: tuple, scaling: tuple, bps: Optional[tuple], norm=None):
    """(dX, dA_g, dB_g, dA_u, dB_u, dA_d, dB_d) of the gated MLP. ``norm`` =
    (inv_rms, weight, offset) when ``x`` is the frozen RMSNorm's input;
    ``adapters`` is (A_g, A_u, A_d)."""
    if bps is None or _off() or not dy.is_cuda:
        return None
    i, h = _rows_cols(qs[0].shape)
    ag, au, ad = adapters
    dev, m, r = dy.get_device(), dy.shape[0], ag.shape[0]
    if not (m > 0 and _rows(dy, dev, m, h) and _rows(x, dev, m, h) and _rows(gate, dev, m, i) and _rows(up, dev, m, i)
            and (hid is None or _rows(hid, dev, m, i)) and _rows(t_gu, dev, m, 2 * r) and _rows(t_d, dev, m, r)
            and _adapter(ag, dev, r, h) and _adapter(au, dev, r, h) and _adapter(ad, dev, r, i)
            and all(p.get_device() == dev for p in bps)):
        return None
    inv = weight = None
    w_dtype, offset = 0, 0.0
    if norm is not None:
        inv, weight, offset = norm[0], norm[1].detach(), float(norm[2])
        if not (_is(inv, _F32, dev) and inv.shape == (m,) and weight.numel() == h and weight.dtype in (_BF16, _F32)
                and _is(weight, weight.dtype, dev)):
            return None
        w_dtype = ops._rn_dtype(weight, "weight")
    ws = _mlp_weights(*packed, qs, dev)
    if ws is None:
        return None
    d = dy.device
    dx, da_gu = _empty(d, _BF16, m, h), _empty(d, _F32, 2 * r, h)
    db_g, db_u, da_d, db_d = _empty(d, _F32, i, r), _empty(d, _F32, i, r), _empty(d, _F32, r, i), _empty(d, _F32, h, r)
    size = ops._workspace("molt_gated_mlp_backward_workspace", m, h, i, r)
    buf = _empty(d, _U8, size)
    ops._call("molt_gated_mlp_backward", dy.data_ptr(), x.data_ptr(), m, *ws, ag.data_ptr(), au.data_ptr(),
              ad.data_ptr(), r, *scaling, *(p.data_ptr() for p in bps), t_gu.data_ptr(), t_d.data_ptr(),
              gate.data_ptr(), up.data_ptr(), ops._ptr(hid), ops._ptr(inv), ops._ptr(weight), w_dtype, offset,
              dx.data_ptr(), da_gu.data_ptr(), db_g.data_ptr(), db_u.data_ptr(), da_d.data_ptr(), db_d.data_ptr(),
              buf.data_ptr(), size, ops._stream(d))
    return dx, da_gu[:r], db_g, da_gu[r:], db_u, da_d, db_d


# ----------------------------------------------- projections of one input
def _stacked_weights(packed, qs, dev: int):
    k = _rows_cols(qs[0].shape)[1]
    ws = (_lib.NF4Weight * len(qs))()
    for j, (p, q) in enumerate(zip(packed, qs)):
        w = _weight(p, q, dev)
        if w is None or w.cols != k or w.block_size != int(qs[0].blocksize) or w.nibble_order != nibble_order(qs[0]):
            return None
        ws[j] = w
        ws[j].code = qs[0].code.data_ptr()    # one table for the stack: the first projection's
    return ws


def stacked_forward(x: Tensor, packed, lora_a, lora_b, qs, lr: int, s: float):
    """(Y, A_stack, packed B_blocks, T, deq(W)^T) of projections of one input
    that carry a gradient."""
    n = len(qs)
    if _off() or x.dim() != 2 or not x.is_cuda or not 1 <= n <= 7:
        return None
    dev, (m, k), r = x.get_device(), x.shape, lora_a[0].shape[0]
    rows = [_rows_cols(q.shape)[0] for q in qs]
    if not (m > 0 and r > 0 and _rows(x, dev, m, k) and all(_adapter(a, dev, r, k) for a in lora_a)
            and all(_adapter(b, dev, rw, r) for b, rw in zip(lora_b, rows))):
        return None
    ws = _stacked_weights(packed, qs, dev)
    if ws is None or ws[0].cols != k:
        return None
    d, total = x.device, sum(rows)
    y, t, a_stack = _empty(d, _BF16, m, total), _empty(d, _BF16, m, lr), _empty(d, _F32, lr, k)
    wt, bp = _empty(d, _BF16, k, total), _packed_b(d, total, lr)
    pa = (C.c_void_p * n)(*[a.data_ptr() for a in lora_a])
    pb = (C.c_void_p * n)(*[b.data_ptr() for b in lora_b])
    written = C.c_int32(0)
    size = ops._workspace("molt_stacked_forward_workspace", m, total, k, lr)
    buf = _empty(d, _U8, size)
    ops._call("molt_stacked_forward", x.data_ptr(), m, n, ws, pa, pb, r, lr, s, a_stack.data_ptr(), bp.data_ptr(),
              t.data_ptr(), y.data_ptr(), wt.data_ptr(), C.byref(written), buf.data_ptr(), size, ops._stream(d))
    return y, a_stack, bp, t, wt if written.value else None


def stacked_backward(dy: Tensor, x: Tensor, t: Tensor, packed, qs, wt: Tensor, a_stack: Tensor, bp: Tensor, r: int,
                     s: float):
    """(dX, dA of the stack, [dB_i]) of projections of one input."""
    n = len(qs)
    if _off() or not dy.is_cuda or not 1 <= n <= 7:
        return None
    dev, (m, k), lr = dy.get_device(), x.shape, t.shape[1]
    rows = [_rows_cols(q.shape)[0] for q in qs]
    total = sum(rows)
    if not (m > 0 and _rows(dy, dev, m, total) and _rows(x, dev, m, k) and _rows(t, dev, m, lr)
            and _rows(wt, dev, k, total) and _adapter(a_stack, dev, lr, k) and bp.get_device() == dev):
        return None
    ws = _stacked_weights(packed, qs, dev)
    if ws is None:
        return None
    d = dy.device
    dx, da = _empty(d, _BF16, m, k), _empty(d, _F32, lr, k)
    dbs = [_empty(d, _F32, rw, r) for rw in rows]
    size = ops._workspace("molt_stacked_backward_workspace", m, n, tuple(rows), k, r, lr)
    buf = _empty(d, _U8, size)
    pdb = (C.c_void_p * n)(*[b.data_ptr() for b in dbs])
    ops._call("molt_stacked_backward", dy.data_ptr(), x.data_ptr(), t.data_ptr(), m, n, ws, wt.data_ptr(),
              a_stack.data_ptr(), bp.data_ptr(), r, lr, s, dx.data_ptr(), da.data_ptr(), pdb, buf.data_ptr(), size,
              ops._stream(d))
    return dx, da, dbs
