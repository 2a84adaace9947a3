"""Fused dequant-attention entry points on the GPU.

Drop-ins for the reference's src/quantization/kernels/fused_dequant_attn.py:301-368
(``fused_dequant_attn_decode``) and :371-435 (``fused_dequant_attn_forward``) with the
numerics of its torch path
(src/quantization/fused_dequant_attn.py:326-331,388-390):
    K = (Kq - zp) * s, V = (Vq - zp) * s, out = softmax(q K^T * sm_scale) V,
sm_scale defaulting to 1/sqrt(head_dim).  Unlike the reference's Triton kernel
(which drops sm_scale and mis-addresses K, see its :69-78,353-365) this computes
exactly that formula, and it also accepts GQA (q heads a multiple of kv heads).

The reference passes unpacked codes (one uint8 per value) with per-token
scales/zps [B, H, S], which the kernels attend as they are: the split-K decode kernel
(hkv_fused_decode) and the MFMA prefill kernel (hkv_fused_forward; where the query rows read
the codes often, they are repacked into block records first).  Calls may run on several streams
at once.  q may be fp16 or bf16 (bf16 is narrowed to fp16 operands exactly within the fp16
range).  Device errors (an out-of-range bf16
value, a decode placement failure) go to a per-device error word that is read without
blocking at the next call -- a later call raises HeteroKVError -- or at once by
check_errors().
"""
import collections
import math
import threading
from typing import Optional

import torch

from . import _lib, ops
from ._lib import HeteroKVError


_ERR = {}   # device -> ErrorWord shared by the calls on that device
_WS = collections.OrderedDict()   # (device, raw stream) -> DecodeWorkspace, the last used at the end
_WS_LIMIT = 32   # the oldest goes beyond that (its memory returns to its own stream's allocator pool)
_AGENT = set()   # devices on which a launch's ranges did not share an XCD: device-scope hand-off
_LOCK = threading.Lock()


def _errword(device):
    with _LOCK:
        w = _ERR.get(device)
        if w is None:
            w = _ERR[device] = ops.ErrorWord(device)
            w.on_error = lambda bits: _placement_failed(device) if bits & _lib.ERR_BIT_PLACEMENT else None
    return w


def _workspace(device, stream):
    """The decode workspace of calls on `device` in `stream` (a raw stream): launches that share
    one are ordered by their stream, so every stream has its own."""
    key = (device, stream)
    with _LOCK:
        ws = _WS.get(key)
        if ws is None:
            ws = _WS[key] = ops.DecodeWorkspace(device, agent_handoff=device in _AGENT)
            while len(_WS) > _WS_LIMIT:
                _WS.popitem(last=False)
        else:
            _WS.move_to_end(key)
    return ws


def _call_workspace(device):
    """This call's workspace.  Under graph capture one of its own: the fill that clears it is
    then part of every replay, and no other call or graph shares it."""
    if torch.cuda.is_current_stream_capturing():
        return ops.DecodeWorkspace(device, agent_handoff=device in _AGENT)
    return _workspace(device, ops.stream_ptr(device).value)


def _placement_failed(device):
    """Tickets of this device's workspaces may be left inconsistent: none is used again (a new
    one is cleared in its own stream), and all launches use the device-scope hand-off."""
    with _LOCK:
        _AGENT.add(device)
        for key in [k for k in _WS if k[0] == device]:
            del _WS[key]


def check_errors(device=None) -> None:
    """Raise HeteroKVError if a call on `device` (default: every device used) reported a
    device error (synchronizes)."""
    for d, w in list(_ERR.items()):
        if device is None or torch.device(device) == d:
            w.check()


def _as_4d(t):
    if t.dim() == 2:
        return t.unsqueeze(0).unsqueeze(0)
    if t.dim() == 3:
        return t.unsqueeze(0)
    return t


def _as_kernel_q(q: torch.Tensor, err) -> torch.Tensor:
    """q in a dtype the kernels take: fp16 and bf16 as they are (the kernels range-check a
    bf16 q themselves); any other floating dtype is rounded to fp16, and a finite value
    beyond the fp16 range (which would become inf) sets HKV_ERR_BIT_RANGE in `err` on the
    device, reported like the kernels' own range errors (no host synchronization)."""
    if q.dtype in (torch.float16, torch.bfloat16):
        return q
    over = (q.abs() > 65504.0) & torch.isfinite(q)
    torch.bitwise_or(err.dev, over.any().to(torch.int32) * _lib.ERR_BIT_RANGE, out=err.dev)
    return q.to(torch.float16)


def fused_dequant_attn_decode(q: torch.Tensor, k_data: torch.Tensor, k_scales: torch.Tensor,
                              k_zps: torch.Tensor, v_data: torch.Tensor, v_scales: torch.Tensor,
                              v_zps: torch.Tensor, sm_scale: Optional[float] = None) -> torch.Tensor:
    """q [B, Hq, 1, D] fp16; k/v_data uint8 [B, Hkv, S, D]; scales/zps [B, Hkv, S] -> [B, Hq, 1, D] in q.dtype."""
    if q.dim() != 4 or q.shape[2] != 1:
        raise HeteroKVError(-1, "Decode expects [B,H,1,D], got %s" % (tuple(q.shape),))
    B, Hq, _, D = q.shape
    kd, vd = _as_4d(k_data), _as_4d(v_data)
    if kd.dim() == 4 and kd.shape[0] != B:
        raise HeteroKVError(-1, "batch mismatch between q and k_data")
    if sm_scale is None:
        sm_scale = 1.0 / math.sqrt(D)
    err = _errword(q.device)
    err.poll()
    qq = _as_kernel_q(q, err)
    out = ops.fused_decode(qq, kd, vd, k_scales, v_scales, k_zps, v_zps, sm_scale,
                           _call_workspace(q.device), err, qq.dtype)
    err.post()
    return out.to(q.dtype)


def fused_dequant_attn_forward(q: torch.Tensor, k_data: torch.Tensor, k_scales: torch.Tensor,
                               k_zps: torch.Tensor, v_data: torch.Tensor, v_scales: torch.Tensor,
                               v_zps: torch.Tensor, sm_scale: Optional[float] = None) -> torch.Tensor:
    """q [B, Hq, Sq, D] fp16/bf16 against quantized K/V [B, Hkv, S, D] (all keys visible,
    as the reference's torch path) -> [B, Hq, Sq, D] in q.dtype."""
    if q.dim() != 4:
        raise HeteroKVError(-1, "Forward expects [B,H,S,D], got %s" % (tuple(q.shape),))
    if sm_scale is None:
        sm_scale = 1.0 / math.sqrt(q.shape[-1])
    err = _errword(q.device)
    err.poll()
    kd, vd = _as_4d(k_data), _as_4d(v_data)
    qq = _as_kernel_q(q, err)
    out = ops.fused_forward(qq, kd, vd, k_scales, v_scales, k_zps, v_zps, sm_scale, err, qq.dtype)
    err.post()
    return out.to(q.dtype)
