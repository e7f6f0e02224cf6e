"""Host wrapper of the prefill-continuation kernel (kernel 3).

Replaces the reference's per-request dense read path for long requests
(oscar_ascend/backend.py:361-415: oscar_full_dequant + _stage_splice +
oscar_prefill / the vendor fused attention op, prefill.py:21-72): causal
attention of the requests' new tokens over their INT2 histories (owner-matched
FP32 window values override) plus themselves, dequantizing history tiles in
LDS; no history is materialised in HBM.
"""
from __future__ import annotations

import ctypes

import torch

from ..format import check_d
from . import _lib, decode, staging
from .quant import cache_geometry


def prefill_continuation(q_rot, k_rot, v_rot, kc, vc, bt_row, cached_len: int, scale: float,
                         stage=None) -> torch.Tensor:
    """q_rot [N, Hq, D], k_rot / v_rot [N, Hk, D] (rotated, any float dtype);
    returns the rotated-V-domain output, fp32 [N, Hq, D]."""
    N, hq, d = q_rot.shape
    check_d(d)
    hk = k_rot.shape[1]
    dev = q_rot.device
    out = torch.empty(N, hq, d, dtype=torch.float32, device=dev)
    if N == 0:
        return out
    q = q_rot.float().contiguous()
    k = k_rot.float().contiguous()
    v = v_rot.float().contiguous()
    bt = bt_row.to(device=dev, dtype=torch.int32).contiguous().reshape(-1)
    bs, pages, kst, vst = cache_geometry(kc, vc)
    if stage is not None:
        sk, sv, owner = stage[:3]
        sk, sv = sk.float().contiguous(), sv.float().contiguous()
        owner = owner.to(torch.int64).contiguous()
        rows = owner.shape[0]
    else:
        sk = sv = owner = None
        rows = 0
    ws = decode.workspace(dev, _lib.load().oscar_prefill_workspace_bytes(N, hq, hk, int(cached_len)))
    _lib.call("oscar_prefill_continuation_split", _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), N, hq, hk, d,
              _lib.ptr(kc), _lib.ptr(vc), bs, pages, *kst, *vst, _lib.ptr(bt), bt.numel(),
              int(cached_len), _lib.ptr(sk), _lib.ptr(sv), _lib.ptr(owner), rows, float(scale),
              _lib.ptr(out), _lib.ptr(ws), ws.numel(), _lib.stream_handle(dev))
    return out


def prefill_rotated(query, key, value, requests, rot_k_op, rot_v_op, rot_vt_op, kc, vc, block_tables, scale: float,
                    out, stage=None) -> None:
    """The long requests of a step, from its bf16 query [N, Hq, D] and key /
    value [N, Hk, D] to rows of its bf16 output [N, Hq, D]: rotations, read and
    output rotation of every request in one call.  requests: (first token,
    new tokens, cached length, block-table row) each; rot_*_op: the rotation
    operands of R_k, R_v and R_v^T."""
    n, hq, d = query.shape
    hk = key.shape[1]
    check_d(d)
    dev = query.device
    for x in (query, key, value, out):
        if x.dtype != torch.bfloat16 or x.device != dev:
            raise ValueError("the rotated prefill takes bf16 query / key / value and writes a bf16 output")
    query, qs = _token_rows(query)
    key, ks = _token_rows(key)
    value, vs = _token_rows(value)
    if ks != vs:
        key, value = key.contiguous(), value.contiguous()
        ks = hk * d
    if not out.is_contiguous() or out.data_ptr() % 16 or tuple(out.shape) != (n, hq, d):
        raise ValueError("the output must be a contiguous, 16-byte aligned [N, Hq, D] tensor")
    rows_bt = block_tables.shape[0]
    for first, new, cached, row in requests:
        if first < 0 or new < 0 or first + new > min(n, key.shape[0], value.shape[0]) or not 0 <= row < rows_bt:
            raise ValueError("a request lies outside the step's tokens or the block table")
    if block_tables.dtype != torch.int32 or block_tables.device != dev or block_tables.stride(1) != 1:
        block_tables = block_tables.to(device=dev, dtype=torch.int32).contiguous()
    bs, pages, kst, vst = cache_geometry(kc, vc)
    sk = sv = owner = None
    rows = 0
    if stage is not None:
        sk, sv, owner = stage[:3]
        rows = staging.check_arena(sk, sv, owner, bs, hk, d)
    B = len(requests)
    first, new = ((ctypes.c_int32 * B)(*[r[i] for r in requests]) for i in (0, 1))
    cached = (ctypes.c_int64 * B)(*[r[2] for r in requests])
    table = (ctypes.c_int32 * B)(*[r[3] for r in requests])
    addr = ctypes.addressof
    ws = decode.workspace(dev, _lib.load().oscar_prefill_rotated_workspace_bytes(B, addr(new), addr(cached), hq, hk))
    _lib.call("oscar_prefill_rotated", _lib.ptr(query), qs, _lib.ptr(key), _lib.ptr(value), ks, B, addr(first),
              addr(new), addr(cached), addr(table), hq, hk, d, _lib.ptr(rot_k_op), _lib.ptr(rot_v_op),
              _lib.ptr(rot_vt_op), _lib.ptr(kc), _lib.ptr(vc), bs, pages, *kst, *vst, _lib.ptr(block_tables),
              block_tables.stride(0), block_tables.shape[1], _lib.ptr(sk), _lib.ptr(sv), _lib.ptr(owner), rows,
              float(scale), _lib.ptr(out), _lib.ptr(ws), ws.numel(), _lib.stream_handle(dev))


def _token_rows(x):
    """x [N, H, D] and its token stride, as rows of H * D contiguous features
    that 16-byte loads can read (a copy where it is none)."""
    n, h, d = x.shape
    if x.stride(2) != 1 or x.stride(1) != d or x.stride(0) % 8 or x.data_ptr() % 16:
        x = x.contiguous()
    return x, x.stride(0) if n > 1 else h * d
