"""ctypes binding of libheterokv.so (declared in include/heterokv.h).

The library is loaded after torch so that it resolves torch's HIP runtime
(same soname) instead of loading a second one.  There is no fallback: if the
library is missing or a call fails, a HeteroKVError is raised.
"""
import ctypes
import os
import threading

import torch  # noqa: F401  (must be loaded before the HIP library, see above)

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libheterokv.so")

ABI_VERSION = 9
DTYPE_F16, DTYPE_BF16, DTYPE_F32, DTYPE_U8 = 0, 1, 2, 3
MAX_F16_ZONES = 3
DECODE_DETERMINISTIC = 1   # HKV_DECODE_DETERMINISTIC
DECODE_AGENT_HANDOFF = 2   # HKV_DECODE_AGENT_HANDOFF
DECODE_SCRATCH_BYTES = 8 << 20   # HKV_DECODE_SCRATCH_BYTES (hkv_decode_attn_noalloc)
BLOCK_TOKENS = 16
HEAD_DIM = 128

HKV_OK = 0
ERR_NAMES = {-1: "HKV_ERR_ARG", -2: "HKV_ERR_HIP", -3: "HKV_ERR_CAPACITY", -4: "HKV_ERR_UNSUPPORTED",
             -5: "HKV_ERR_DEVICE"}
ERR_DEVICE = -5   # HKV_ERR_DEVICE: a device error word came back non-zero

# device error-word bits (HKV_ERR_BIT_*)
ERR_BIT_BLOCK_ID, ERR_BIT_SLOT, ERR_BIT_PLACEMENT, ERR_BIT_RANGE = 1, 2, 4, 8
_ERR_BIT_TEXT = {
    ERR_BIT_BLOCK_ID: "a block table held an id outside the pool / staging records",
    ERR_BIT_SLOT: "a token slot lay beyond its block table row",
    ERR_BIT_PLACEMENT: "decode ranges of one (sequence, kv head) ran on more than one XCD; that launch's "
                       "output is invalid (later launches use the device-scope hand-off)",
    ERR_BIT_RANGE: "a finite bf16 or fp32 value beyond the fp16 range (|x| > 65504) was narrowed to fp16",
}


def describe_error_bits(bits):
    """Human-readable text of a device error word."""
    parts = [t for b, t in sorted(_ERR_BIT_TEXT.items()) if bits & b]
    unknown = bits & ~sum(_ERR_BIT_TEXT)
    if unknown:
        parts.append("unknown error bits 0x%x" % unknown)
    return "; ".join(parts)


class HeteroKVError(RuntimeError):
    """A libheterokv call failed (carries the C return code)."""

    def __init__(self, code, msg):
        super().__init__("%s (%d): %s" % (ERR_NAMES.get(code, "HKV_ERR"), code, msg))
        self.code = code


vp = ctypes.c_void_p
i32 = ctypes.c_int32
i64 = ctypes.c_int64


class PackArgs(ctypes.Structure):
    _fields_ = [("k", vp), ("v", vp), ("dtype", i32),
                ("src_stride_b", i64), ("src_stride_h", i64), ("src_stride_t", i64),
                ("batch", i32), ("num_kv_heads", i32), ("head_dim", i32), ("num_tokens", i32),
                ("start_pos", vp), ("block_table", vp), ("bt_stride", i32),
                ("pool", vp), ("pool_blocks", i64), ("err_flag", vp), ("start_base", i32)]


class RepackArgs(ctypes.Structure):
    _fields_ = [("k_codes", vp), ("v_codes", vp),
                ("code_stride_b", i64), ("code_stride_h", i64), ("code_stride_t", i64),
                ("k_scales", vp), ("v_scales", vp), ("k_zps", vp), ("v_zps", vp), ("zp_dtype", i32),
                ("meta_stride_b", i64), ("meta_stride_h", i64), ("meta_stride_t", i64),
                ("batch", i32), ("num_kv_heads", i32), ("head_dim", i32), ("num_tokens", i32),
                ("start_pos", vp), ("block_table", vp), ("bt_stride", i32),
                ("pool", vp), ("pool_blocks", i64), ("err_flag", vp)]


class ZoneWriteArgs(ctypes.Structure):
    _fields_ = [("k", vp), ("v", vp),
                ("src_stride_b", i64), ("src_stride_h", i64), ("src_stride_t", i64),
                ("batch", i32), ("num_kv_heads", i32), ("head_dim", i32), ("num_tokens", i32),
                ("slot_start", vp), ("capacity", i32), ("ring", i32),
                ("zone_k", vp), ("zone_v", vp), ("slot_base", i32), ("dtype", i32), ("err_flag", vp)]


class ZoneStepArgs(ctypes.Structure):
    _fields_ = [("k", vp), ("v", vp), ("src_stride_b", i64), ("src_stride_h", i64),
                ("batch", i32), ("num_kv_heads", i32), ("head_dim", i32),
                ("tail_k", vp), ("tail_v", vp), ("tail_capacity", i32), ("tail_ring", i32),
                ("hh_k", vp), ("hh_v", vp), ("hh_capacity", i32), ("hh_budget", i32),
                ("state", vp), ("tail_lens", vp), ("hh_lens", vp), ("dtype", i32), ("err_flag", vp)]


class F16Zone(ctypes.Structure):
    _fields_ = [("k", vp), ("v", vp), ("capacity", i32), ("max_len", i32), ("lens", vp)]


class DecodeArgs(ctypes.Structure):
    _fields_ = [("batch", i32), ("num_q_heads", i32), ("num_kv_heads", i32), ("head_dim", i32),
                ("sm_scale", ctypes.c_float),
                ("q", vp), ("q_stride_b", i64), ("q_stride_h", i64),
                ("num_f16_zones", i32), ("f16", F16Zone * MAX_F16_ZONES),
                ("pool", vp), ("pool_blocks", i64), ("block_table", vp), ("bt_stride", i32),
                ("int4_lens", vp), ("int4_max_len", i32),
                ("out", vp), ("out_stride_b", i64), ("out_stride_h", i64),
                ("workspace", vp), ("workspace_bytes", ctypes.c_size_t), ("splits_hint", i32),
                ("staging", vp), ("staging_blocks", i64), ("flags", i32),
                ("scores", vp), ("scores_stride_b", i64), ("scores_stride_h", i64), ("score_stats", vp),
                ("q_dtype", i32), ("out_dtype", i32), ("err_flag", vp)]


class PrefillArgs(ctypes.Structure):
    _fields_ = [("batch", i32), ("num_q_heads", i32), ("num_kv_heads", i32), ("head_dim", i32),
                ("num_queries", i32), ("sm_scale", ctypes.c_float),
                ("q", vp), ("q_stride_b", i64), ("q_stride_h", i64), ("q_stride_t", i64),
                ("num_f16_zones", i32), ("f16", F16Zone * MAX_F16_ZONES),
                ("pool", vp), ("pool_blocks", i64), ("block_table", vp), ("bt_stride", i32),
                ("int4_lens", vp), ("int4_max_len", i32),
                ("chunk_k", vp), ("chunk_v", vp),
                ("chunk_stride_b", i64), ("chunk_stride_h", i64), ("chunk_stride_t", i64),
                ("out", vp), ("out_stride_b", i64), ("out_stride_h", i64), ("out_stride_t", i64),
                ("err_flag", vp), ("staging", vp), ("staging_blocks", i64),
                ("q_dtype", i32), ("chunk_dtype", i32), ("out_dtype", i32),
                ("workspace", vp), ("workspace_bytes", ctypes.c_size_t)]


class FusedArgs(ctypes.Structure):
    _fields_ = [("batch", i32), ("num_q_heads", i32), ("num_kv_heads", i32), ("head_dim", i32),
                ("num_queries", i32), ("num_tokens", i32), ("sm_scale", ctypes.c_float),
                ("q_dtype", i32), ("out_dtype", i32), ("flags", i32),
                ("q", vp), ("q_stride_b", i64), ("q_stride_h", i64), ("q_stride_t", i64),
                ("k_codes", vp), ("v_codes", vp), ("k_scales", vp), ("v_scales", vp), ("k_zps", vp), ("v_zps", vp),
                ("out", vp), ("out_stride_b", i64), ("out_stride_h", i64), ("out_stride_t", i64),
                ("err_flag", vp), ("workspace", vp), ("workspace_bytes", ctypes.c_size_t)]


class CopyDesc(ctypes.Structure):
    _fields_ = [("dst", vp), ("src", vp), ("bytes", ctypes.c_size_t)]


class PfStats(ctypes.Structure):
    _fields_ = [("bytes_h2d", ctypes.c_uint64), ("copies_h2d", ctypes.c_uint64),
                ("bytes_d2h", ctypes.c_uint64), ("arena_bytes", ctypes.c_uint64)]


# (name, restype, argtypes) of every symbol include/heterokv.h declares.
SYMBOLS = [
    ("hkv_abi_version", ctypes.c_int, []),
    ("hkv_last_error", ctypes.c_char_p, []),
    ("hkv_block_bytes", i64, [i32, i32]),
    ("hkv_quantize_groups", ctypes.c_int, [vp, i32, i64, i32, vp, vp, vp, vp]),
    ("hkv_dequantize_groups", ctypes.c_int, [vp, vp, vp, i64, i32, vp, i32, vp]),
    ("hkv_pack_tokens", ctypes.c_int, [ctypes.POINTER(PackArgs), vp]),
    ("hkv_repack_codes", ctypes.c_int, [ctypes.POINTER(RepackArgs), vp]),
    ("hkv_unpack_tokens", ctypes.c_int, [vp, i64, vp, i32, i32, i32, i32, vp, vp, vp, vp]),
    ("hkv_dequant_tokens", ctypes.c_int, [vp, i64, vp, i32, i32, i32, i32, i32, vp, vp, i32, vp]),
    ("hkv_zone_write", ctypes.c_int, [ctypes.POINTER(ZoneWriteArgs), vp]),
    ("hkv_zone_read", ctypes.c_int, [vp, vp, i32, i32, i32, i32, i32, vp, vp, vp]),
    ("hkv_zone_copy", ctypes.c_int, [vp, vp, i32, i32, vp, vp, i32, i32, i32, i32, i32, i32, vp]),
    ("hkv_zone_step", ctypes.c_int, [ctypes.POINTER(ZoneStepArgs), vp]),
    ("hkv_decode_workspace_bytes", ctypes.c_size_t, [i32, i32, i32, i32, i32, vp, i32]),
    ("hkv_decode_attn", ctypes.c_int, [ctypes.POINTER(DecodeArgs), vp]),
    ("hkv_decode_ranges", ctypes.c_int, [ctypes.POINTER(DecodeArgs), ctypes.POINTER(i32)]),
    ("hkv_decode_attn_noalloc", ctypes.c_int, [ctypes.POINTER(DecodeArgs), vp]),
    ("hkv_prefill_workspace_bytes", ctypes.c_size_t, [i32, i32, i32]),
    ("hkv_prefill_split_bytes", ctypes.c_size_t, [ctypes.POINTER(PrefillArgs)]),
    ("hkv_prefill_attn", ctypes.c_int, [ctypes.POINTER(PrefillArgs), vp]),
    ("hkv_fused_decode", ctypes.c_int, [ctypes.POINTER(FusedArgs), vp]),
    ("hkv_fused_forward", ctypes.c_int, [ctypes.POINTER(FusedArgs), vp]),
    ("hkv_fused_forward_workspace_bytes", ctypes.c_size_t, [ctypes.POINTER(FusedArgs)]),
    ("hkv_pf_create", ctypes.c_int, [i32, ctypes.c_size_t, i32, ctypes.POINTER(vp)]),
    ("hkv_pf_destroy", ctypes.c_int, [vp]),
    ("hkv_pf_host_ptr", vp, [vp, ctypes.c_size_t]),
    ("hkv_pf_stream", vp, [vp]),
    ("hkv_pf_stage_out", ctypes.c_int, [vp, vp, ctypes.c_size_t, ctypes.c_size_t, vp]),
    ("hkv_pf_submit", ctypes.c_int, [vp, ctypes.POINTER(CopyDesc), i32, i32, i32]),
    ("hkv_pf_record", ctypes.c_int, [vp, i32]),
    ("hkv_pf_wait", ctypes.c_int, [vp, i32, vp]),
    ("hkv_pf_mark", ctypes.c_int, [vp, i32, vp]),
    ("hkv_pf_stall_ms", ctypes.c_int, [vp, i32, ctypes.POINTER(ctypes.c_float)]),
    ("hkv_pf_stats", ctypes.c_int, [vp, ctypes.POINTER(PfStats)]),
    ("hkv_pf_synchronize", ctypes.c_int, [vp]),
    ("hkv_gather_blocks", ctypes.c_int, [vp, i64, vp, i64, vp, i64, i64, vp, vp, vp]),
    ("hkv_attn_weights", ctypes.c_int, [vp, i64, i64, vp, i32, i32, i64, vp, vp, i64, i32, vp]),
    ("hkv_block_scores", ctypes.c_int, [vp, i64, i32, vp, vp]),
    ("hkv_eviction_workspace_bytes", ctypes.c_size_t, [i64, i32, i32, i32, i32]),
    ("hkv_eviction_candidates", ctypes.c_int, [vp, i64, i32, i32, i32, i32, vp, ctypes.POINTER(i32), vp,
                                                ctypes.c_size_t, vp]),
]

_lock = threading.Lock()
_lib = None


def load():
    """Load libheterokv.so once; raises if it is missing or has the wrong ABI."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(LIB_PATH):
            raise HeteroKVError(-2, "libheterokv.so not built at %s (run __graft_entry__.build() or "
                                    "hetero-kvcache-optimizer_amd/build.py)" % LIB_PATH)
        lib = ctypes.CDLL(LIB_PATH)
        for name, res, args in SYMBOLS:
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        ver = lib.hkv_abi_version()
        if ver != ABI_VERSION:
            raise HeteroKVError(-1, "libheterokv ABI %d, expected %d" % (ver, ABI_VERSION))
        _lib = lib
    return _lib


def check(rc, what=""):
    if rc != HKV_OK:
        msg = load().hkv_last_error().decode("utf-8", "replace")
        raise HeteroKVError(rc, (what + ": " if what else "") + msg)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_ptr(device=None):
    """Raw hipStream_t of torch's current stream on `device` (a torch.device, an index or
    None for the current device)."""
    if _raw_stream is not None:
        if isinstance(device, torch.device):
            idx = device.index if device.index is not None else torch.cuda.current_device()
        elif isinstance(device, int):
            idx = device
        elif device is None:
            idx = torch.cuda.current_device()
        else:
            d = torch.device(device)
            idx = d.index if d.index is not None else torch.cuda.current_device()
        return ctypes.c_void_p(_raw_stream(idx))
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)
