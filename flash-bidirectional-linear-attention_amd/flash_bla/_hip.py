"""Binding of libfbla_hip.so (declared in include/flash_bla_hip.h).

The operators' calls are native (csrc/fbla_torch.cpp, built as _lib/fbla_torch.so): PyTorch is used for device memory
(outputs, state, workspace come from its caching allocator) and for the current stream; all arithmetic happens inside the
library.  `lib()` is the library itself through ctypes.  There is no fallback: a missing library or a non-GPU tensor raises.

    la_fwd(q, k, v, q_rope, k_rope, scale, eps, flags) -> o, s, km          dense [B, H, L, D]; k, v of any length
    la_bwd(q, k, v, q_rope, k_rope, do, s, km, scale, eps, flags) -> dq, dk, dv, dq_rope, dk_rope
    pair_supported(q, v), pair_fwd(q1, q2, k, v, scale, eps) -> o1, o2, s, km
    pair_bwd(q1, q2, k, v, do1, do2, s, km, scale, eps) -> dq1, dq2, dk, dv
    varlen_fwd(q, k, v, cu_seqlens, max_seqlen, scale, eps, extra_flags=0) -> o, s, km      packed [T, H, D]
    varlen_bwd(q, k, v, cu_seqlens, max_seqlen, do, s, km, scale, eps, extra_flags=0) -> dq, dk, dv
    chunk_reduce(q, k, v, chunk, with_norm=False, p_norm=2.0) -> qc, kc, vc, h, h_norm or None      fp32
    select_blocks(qc, kc, bias, top_k, scale) -> int32 indices, ascending
    piecewise_supported(q, v, block), piecewise_fwd(q, k, v, kc, vc, h, indices, block, scale) -> o
    elu1_fwd(x0, x1=None) -> y0 or (y0, y1), elu1_bwd(x, dy) -> dx
    dwconv_fwd(x, w, bias, H, W, flip=False) -> y, dwconv_grad(x, g, w, H, W, with_bias) -> dw, db
    linear_wgrad(g, x, with_bias) -> dw, db
    project([(a, w, bias, add, a2, w2), ...], rows_of_w) -> [a w^T + bias + add, ...] or (rows_of_w) [a w + a2 w2 + add, ...]
    projects(x, w, alone) -> whether a whole block runs a product of these rows on `project` (and not on the library's GEMM)
    norm_leaky([(x, weight, bias, eps, slope), ...], with_stats) -> [(y, mean, rstd), ...]
    polarity_fwd(qg, kv, pe, scale, power, heads) -> q_same, q_opp, k_both, v
    polarity_bwd(qg, kv, pe, scale, power, heads, dq_same, dq_opp, dk_both, dv, dv_rows, dgate) -> dqg, dkv, dpe, dscale, dpower
    rotary_fwd(qk, x, rotations, heads) -> q, k, q_rot, k_rot, v
    rotary_bwd(qk, rotations, heads, dq, dk, dq_rot, dk_rot, dv, dv_rows) -> dqk, dx
    merge_fwd(o, o2, local, gate) -> rows, merge_bwd(dout, heads, halves, o, o2, local, gate) -> do, do2, dlocal, dgate
    interpolate_fwd(x, tokens) -> y, interpolate_bwd(g, n) -> dx
    focus_fwd(q, kv, pe, scale, heads) -> q, k, v
    focus_bwd(q, kv, pe, scale, heads, dq_heads, dk_heads, dv_heads, dv_rows) -> dq, dkv, dpe, dscale
    turn_fwd(q, k, weight, rotations) -> k * weight, q turned, k * weight turned
    turn_bwd(k, weight, rotations, dk_out, dq_rot, dk_rot) -> dq, dk, dweight

Whole blocks (layers/_whole.py) and the checks in front of them: mlla_*, pola_*, focused_*, linfusion_*, plain_gpu_tensors,
untouched_modules, dense_operands.

Tensors that are not contiguous or off a 16-byte boundary are copied first.
"""
import ctypes
import importlib.util
import os
import threading

import torch

# FBLA_LIB_PATH selects another build of the library (A/B comparisons of kernel changes).
_LIB_PATH = os.environ.get("FBLA_LIB_PATH") or os.path.join(
    os.path.dirname(os.path.abspath(__file__)), "_lib", "libfbla_hip.so")
_lib = None

F16, BF16, F32 = 0, 1, 2
NORMALIZE, DECOUPLED, DEFAULT_SCALE, ELU1_QK, ELU1_GRAD = 1, 2, 4, 8, 16

_DTYPES = {torch.float16: F16, torch.bfloat16: BF16, torch.float32: F32}

_vp, _i64, _i32, _f32, _sz = (ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float,
                              ctypes.c_size_t)

_SIGNATURES = {
    "fbla_version": (ctypes.c_int, []),
    "fbla_last_error": (ctypes.c_char_p, []),
    "fbla_set_phase_mask": (None, [ctypes.c_uint]),
    "fbla_la_workspace_bytes": (_sz, [_i32, _i64, _i64, _i64, _i32, _i32, _i32, _i32]),
    "fbla_la_fwd": (_i32, [_vp] * 9 + [_sz, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_static_scratch_bytes": (_sz, []),
    "fbla_la_fwd_static": (_i32, [_vp] * 8 + [_i64, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_la_bwd": (_i32, [_vp] * 14 + [_sz, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_la_pair_workspace_bytes": (_sz, [_i32, _i64, _i64, _i64, _i32, _i32, _i32]),
    "fbla_la_pair_fwd": (_i32, [_vp] * 9 + [_sz, _i64, _i64, _i64, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_la_pair_bwd": (_i32, [_vp] * 13 + [_sz, _i64, _i64, _i64, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_la_cross_workspace_bytes": (_sz, [_i32, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _i32]),
    "fbla_la_cross_fwd": (_i32, [_vp] * 7 + [_sz, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_la_cross_bwd": (_i32, [_vp] * 10 + [_sz, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_decoupled_cross_fwd": (_i32, [_vp] * 9 + [_sz, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_decoupled_cross_bwd": (_i32, [_vp] * 14 + [_sz, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_varlen_workspace_bytes": (_sz, [_i32, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _i32]),
    "fbla_varlen_fwd": (_i32, [_vp] * 8 + [_sz, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_varlen_bwd": (_i32, [_vp] * 11 + [_sz, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _f32, _vp]),
    "fbla_chunk_reduce_workspace_bytes": (_sz, [_i64, _i64, _i32, _i32, _i32, _i32, _i32]),
    "fbla_chunk_reduce": (_i32, [_vp] * 9 + [_sz, _i64, _i64, _i32, _i32, _i32, _f32, _i32, _vp]),
    "fbla_select_blocks": (_i32, [_vp] * 4 + [_i64, _i64, _i32, _i32, _f32, _vp]),
    "fbla_piecewise_workspace_bytes": (_sz, [_i64, _i64, _i32, _i32, _i32, _i32]),
    "fbla_piecewise_fwd": (_i32, [_vp] * 9 + [_sz, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _i32, _vp]),
    "fbla_elu1_fwd": (_i32, [_vp, _vp, _i64, _vp, _vp, _i64, _i32, _vp]),
    "fbla_elu1_bwd": (_i32, [_vp, _vp, _vp, _i64, _i32, _vp]),
    "fbla_dwconv_fwd": (_i32, [_vp, _i64, _i64, _vp, _vp, _vp] + [_i64] * 5 + [_i32] * 5 + [_vp]),
    "fbla_dwconv_grad_workspace_bytes": (_sz, [_i64] * 3 + [_i32] * 4),
    "fbla_dwconv_grad": (_i32, [_vp, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _vp, _sz] + [_i64] * 3 + [_i32] * 4 + [_vp]),
    "fbla_linear_wgrad_workspace_bytes": (_sz, [_i64] + [_i32] * 3),
    "fbla_linear_wgrad": (_i32, [_vp, _i64, _vp, _i64, _vp, _vp, _vp, _sz, _i64] + [_i32] * 3 + [_vp]),
    "fbla_project": (_i32, [_vp, _i32, _i64, _i32, _i32, _vp]),
    "fbla_norm_leaky": (_i32, [_vp, _i32, _i64, _i32, _i32, _vp]),
    "fbla_polarity_fwd": (_i32, [_vp] * 9 + [_i64] * 3 + [_i32] * 3 + [_vp]),
    "fbla_polarity_bwd_workspace_bytes": (_sz, [_i64] * 3 + [_i32] * 3),
    "fbla_polarity_bwd": (_i32, [_vp] * 17 + [_sz] + [_i64] * 3 + [_i32] * 3 + [_vp]),
    "fbla_rotary_fwd": (_i32, [_vp] * 3 + [_i32] + [_vp] * 5 + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_rotary_bwd": (_i32, [_vp] * 2 + [_i32] + [_vp] * 8 + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_merge_fwd": (_i32, [_vp] * 4 + [_i64, _vp] + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_merge_bwd": (_i32, [_vp] * 5 + [_i64] + [_vp] * 4 + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_block_attn_workspace_bytes": (_sz, [_i32] + [_i64] * 3 + [_i32]),
    "fbla_block_attn_state_elements": (_sz, [_i32, _i64, _i32]),
    "fbla_block_attn_forward": (_i32, [_vp, _vp]),
    "fbla_block_attn_backward_queries": (_i32, [_vp, _vp]),
    "fbla_block_attn_backward_keys": (_i32, [_vp, _vp]),
    "fbla_turn_fwd": (_i32, [_vp] * 7 + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_turn_bwd": (_i32, [_vp] * 9 + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_focus_fwd": (_i32, [_vp] * 7 + [_i64] * 3 + [_i32] * 3 + [_vp]),
    "fbla_focus_bwd_workspace_bytes": (_sz, [_i64] * 3 + [_i32] * 3),
    "fbla_focus_bwd": (_i32, [_vp] * 13 + [_sz] + [_i64] * 3 + [_i32] * 3 + [_vp]),
    "fbla_interpolate_fwd": (_i32, [_vp, _i64, _i64, _vp] + [_i64] * 3 + [_i32] * 2 + [_vp]),
    "fbla_interpolate_bwd": (_i32, [_vp] * 2 + [_i64] * 3 + [_i32] * 2 + [_vp]),
}


def lib_path():
    return _LIB_PATH


def exported_symbols():
    """Names this binding expects the shared library to export."""
    return sorted(_SIGNATURES)


def lib():
    """Load libfbla_hip.so once; raise if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(_LIB_PATH):
            raise RuntimeError(
                f"flash_bla: HIP library not found at {_LIB_PATH}; build it with "
                "`make -C flash-bidirectional-linear-attention_amd/csrc` (there is no fallback path)")
        handle = ctypes.CDLL(_LIB_PATH)
        for name, (restype, argtypes) in _SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = restype
            fn.argtypes = argtypes
        _lib = handle
    return _lib


_NATIVE = frozenset((
    "la_fwd", "la_bwd", "pair_supported", "pair_fwd", "pair_bwd", "varlen_fwd", "varlen_bwd", "chunk_reduce", "select_blocks",
    "piecewise_supported", "piecewise_fwd", "elu1_fwd", "elu1_bwd", "dwconv_fwd", "dwconv_grad", "linear_wgrad", "project", "norm_leaky", "polarity_fwd",
    "polarity_bwd", "rotary_fwd", "rotary_bwd", "merge_fwd", "merge_bwd", "interpolate_fwd", "interpolate_bwd", "focus_fwd",
    "focus_bwd", "turn_fwd", "turn_bwd", "mlla_fwd", "mlla_bwd", "pola_fwd", "pola_bwd", "focused_fwd", "focused_bwd",
    "linfusion_fwd", "linfusion_bwd", "dense_operands", "plain_gpu_tensors", "untouched_modules", "projects", "mlla_fits", "pola_fits",
    "focused_fits", "linfusion_fits"))


_native_lock = threading.Lock()
_native = None


def _load_native():
    global _native
    with _native_lock:  # (once: native calls do not hold the interpreter's lock)
        if _native is None:
            _native = _open_native()
    return _native


def _open_native():
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_lib", "fbla_torch.so")
    if not os.path.exists(path):
        raise RuntimeError(f"flash_bla: host library not found at {path}; build it with "
                           "`make -C flash-bidirectional-linear-attention_amd/csrc` (there is no fallback path)")
    lib()  # (its own message if it is missing)
    spec = importlib.util.spec_from_file_location("fbla_torch", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    module.load(_LIB_PATH)
    return module


def __getattr__(name):
    """The native calls, bound as names of this module when the first of them is asked for."""
    if name not in _NATIVE:
        raise AttributeError(f"module {__name__!r} has no attribute {name!r}")
    module = _load_native()
    for n in _NATIVE:
        globals().setdefault(n, getattr(module, n))
    return globals()[name]


def dtype_code(t):
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise TypeError("q, k, and v must have dtype float16, bfloat16, or float32") from None


def most_row_channels(t):
    """The widest row of t's type that focus_fwd takes."""
    return 4096 // t.element_size()
