"""ctypes binding of libfbla_hip.so (declared in include/flash_bla_hip.h).

PyTorch is used for device memory (outputs, state, workspace come from its
caching allocator) and for the current stream; all arithmetic happens inside the
library.  There is no fallback: a missing library or a non-GPU tensor raises.
"""
import ctypes
import os

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
    "fbla_polarity_fwd": (_i32, [_vp] * 9 + [_i64] * 3 + [_i32] * 3 + [_vp]),
    "fbla_polarity_bwd_workspace_bytes": (_sz, [_i64] * 3 + [_i32] * 3),
    "fbla_polarity_bwd": (_i32, [_vp] * 17 + [_sz] + [_i64] * 3 + [_i32] * 3 + [_vp]),
    "fbla_rotary_fwd": (_i32, [_vp] * 3 + [_i32] + [_vp] * 5 + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_rotary_bwd": (_i32, [_vp] * 2 + [_i32] + [_vp] * 8 + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_merge_fwd": (_i32, [_vp] * 4 + [_i64, _vp] + [_i64] * 2 + [_i32] * 3 + [_vp]),
    "fbla_merge_bwd": (_i32, [_vp] * 5 + [_i64] + [_vp] * 4 + [_i64] * 2 + [_i32] * 3 + [_vp]),
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


def _check(rc, what):
    if rc != 0:
        msg = lib().fbla_last_error().decode("utf-8", "replace")
        exc = ValueError if rc in (-1, -2) else RuntimeError
        raise exc(f"{what} failed ({rc}): {msg}")


def dtype_code(t):
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise TypeError("q, k, and v must have dtype float16, bfloat16, or float32") from None


def _ptr(t):
    return None if t is None else t.data_ptr()


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(device):
    """Handle of torch's current stream on `device` (the raw getter saves the Stream object: these
    wrappers are on the host-bound path of small problems)."""
    if _raw_stream is not None and device.index is not None:
        return _raw_stream(device.index)
    return torch.cuda.current_stream(device).cuda_stream


class _Here:
    """No-op context: the tensors' device is already the current one."""
    def __enter__(self):
        return self

    def __exit__(self, *exc):
        return False


_HERE = _Here()


_one_device = None


def _on(device):
    """Context that makes `device` current for the launch (kernels run on the current device).
    With a single visible GPU there is nothing to switch (and asking torch for the current device
    costs 2 us on the host-bound path of small problems)."""
    global _one_device
    if _one_device is None:
        _one_device = torch.cuda.device_count() == 1
    if _one_device or device.index is None or device.index == torch.cuda.current_device():
        return _HERE
    return torch.cuda.device(device)


def _workspace(nbytes, device):
    return torch.empty(max(int(nbytes), 1), dtype=torch.uint8, device=device)


def _aligned(*tensors):
    """The kernels move 16-byte pieces: a tensor whose storage offset leaves its first element off
    a 16-byte boundary (a view into a larger buffer) is copied to fresh, aligned memory."""
    return tuple(t if t is None or t.data_ptr() % 16 == 0 else t.clone(memory_format=torch.contiguous_format)
                 for t in tensors)


def _require_gpu(*tensors):
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise ValueError("flash_bla HIP operators need GPU tensors (got a CPU tensor); "
                             "use the naive_* functions for CPU math")


def la_fwd(q, k, v, q_rope, k_rope, scale, eps, flags):
    """Dense forward: returns (o, s, km).  Tensors must be contiguous [B,H,L,D]; k and v may have
    another number of tokens than q (not with the decoupled operator)."""
    _require_gpu(q, k, v, q_rope, k_rope)
    q, k, v, q_rope, k_rope = _aligned(q, k, v, q_rope, k_rope)
    L = lib()
    B, H, T, DK = q.shape
    Tk, DV = k.shape[-2], v.shape[-1]
    code = dtype_code(q)
    dev = q.device
    o = torch.empty(B, H, T, DV, dtype=v.dtype, device=dev)
    s = torch.empty(B, H, DK, DV, dtype=torch.float32, device=dev)
    km = torch.empty(B, H, DK, dtype=torch.float32, device=dev)
    if Tk != T and flags & DECOUPLED:
        with _on(dev):
            ws = _workspace(L.fbla_la_cross_workspace_bytes(0, B, H, T, Tk, DK, DV, code, flags), dev)
            rc = L.fbla_decoupled_cross_fwd(_ptr(q), _ptr(k), _ptr(q_rope), _ptr(k_rope), _ptr(v), _ptr(o), _ptr(s),
                                            _ptr(km), _ptr(ws), ws.numel(), B, H, T, Tk, DK, DV, code, float(scale),
                                            float(eps), _stream(dev))
        _check(rc, "fbla_decoupled_cross_fwd")
        return o, s, km
    if Tk != T:
        with _on(dev):
            ws = _workspace(L.fbla_la_cross_workspace_bytes(0, B, H, T, Tk, DK, DV, code, flags), dev)
            rc = L.fbla_la_cross_fwd(_ptr(q), _ptr(k), _ptr(v), _ptr(o), _ptr(s), _ptr(km), _ptr(ws),
                                     ws.numel(), B, H, T, Tk, DK, DV, code, flags, float(scale), float(eps),
                                     _stream(dev))
        _check(rc, "fbla_la_cross_fwd")
        return o, s, km
    with _on(dev):
        ws = _workspace(L.fbla_la_workspace_bytes(0, B, H, T, DK, DV, code, flags), dev)
        rc = L.fbla_la_fwd(_ptr(q), _ptr(k), _ptr(v), _ptr(q_rope), _ptr(k_rope), _ptr(o), _ptr(s),
                           _ptr(km), _ptr(ws), ws.numel(), B, H, T, DK, DV, code, flags,
                           float(scale), float(eps), _stream(dev))
    _check(rc, "fbla_la_fwd")
    return o, s, km


def la_bwd(q, k, v, q_rope, k_rope, do, s, km, scale, eps, flags):
    """Dense backward: returns (dq, dk, dv, dq_rope, dk_rope)."""
    _require_gpu(q, k, v, do)
    q, k, v, q_rope, k_rope, do, s, km = _aligned(q, k, v, q_rope, k_rope, do, s, km)
    L = lib()
    B, H, T, DK = q.shape
    Tk, DV = k.shape[-2], v.shape[-1]
    code = dtype_code(q)
    dev = q.device
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    dqr = torch.empty_like(q_rope) if flags & DECOUPLED else None
    dkr = torch.empty_like(k_rope) if flags & DECOUPLED else None
    if Tk != T and flags & DECOUPLED:
        with _on(dev):
            ws = _workspace(L.fbla_la_cross_workspace_bytes(1, B, H, T, Tk, DK, DV, code, flags), dev)
            rc = L.fbla_decoupled_cross_bwd(_ptr(q), _ptr(k), _ptr(q_rope), _ptr(k_rope), _ptr(v), _ptr(do), _ptr(s),
                                            _ptr(km), _ptr(dq), _ptr(dk), _ptr(dqr), _ptr(dkr), _ptr(dv), _ptr(ws),
                                            ws.numel(), B, H, T, Tk, DK, DV, code, float(scale), float(eps),
                                            _stream(dev))
        _check(rc, "fbla_decoupled_cross_bwd")
        return dq, dk, dv, dqr, dkr
    if Tk != T:
        with _on(dev):
            ws = _workspace(L.fbla_la_cross_workspace_bytes(1, B, H, T, Tk, DK, DV, code, flags), dev)
            rc = L.fbla_la_cross_bwd(_ptr(q), _ptr(k), _ptr(v), _ptr(do), _ptr(s), _ptr(km), _ptr(dq),
                                     _ptr(dk), _ptr(dv), _ptr(ws), ws.numel(), B, H, T, Tk, DK, DV, code,
                                     flags, float(scale), float(eps), _stream(dev))
        _check(rc, "fbla_la_cross_bwd")
        return dq, dk, dv, None, None
    with _on(dev):
        ws = _workspace(L.fbla_la_workspace_bytes(1, B, H, T, DK, DV, code, flags), dev)
        rc = L.fbla_la_bwd(_ptr(q), _ptr(k), _ptr(v), _ptr(q_rope), _ptr(k_rope), _ptr(do), _ptr(s),
                           _ptr(km), _ptr(dq), _ptr(dk), _ptr(dv), _ptr(dqr), _ptr(dkr), _ptr(ws),
                           ws.numel(), B, H, T, DK, DV, code, flags, float(scale), float(eps),
                           _stream(dev))
    _check(rc, "fbla_la_bwd")
    return dq, dk, dv, dqr, dkr


def pair_supported(q, v):
    """Whether the two-query operator covers these shapes (contiguous [B,H,L,DK] / [B,H,L,DV])."""
    B, H, T, DK = q.shape
    return bool(q.is_cuda and q.dtype in (torch.float16, torch.bfloat16) and
                lib().fbla_la_pair_workspace_bytes(0, B, H, T, DK, v.shape[-1], dtype_code(q)))


def pair_fwd(q1, q2, k, v, scale, eps):
    """Two queries on shared keys and values: returns (o1, o2, s, km); o_i are [B,H,L,DV/2]."""
    _require_gpu(q1, q2, k, v)
    q1, q2, k, v = _aligned(q1, q2, k, v)
    L = lib()
    B, H, T, DK = q1.shape
    DV = v.shape[-1]
    code = dtype_code(q1)
    dev = q1.device
    o1 = torch.empty(B, H, T, DV // 2, dtype=v.dtype, device=dev)
    o2 = torch.empty_like(o1)
    s = torch.empty(B, H, DK, DV, dtype=torch.float32, device=dev)
    km = torch.empty(B, H, DK, dtype=torch.float32, device=dev)
    with _on(dev):
        ws = _workspace(L.fbla_la_pair_workspace_bytes(0, B, H, T, DK, DV, code), dev)
        rc = L.fbla_la_pair_fwd(_ptr(q1), _ptr(q2), _ptr(k), _ptr(v), _ptr(o1), _ptr(o2), _ptr(s), _ptr(km),
                                _ptr(ws), ws.numel(), B, H, T, DK, DV, code, float(scale), float(eps), _stream(dev))
    _check(rc, "fbla_la_pair_fwd")
    return o1, o2, s, km


def pair_bwd(q1, q2, k, v, do1, do2, s, km, scale, eps):
    """Backward of pair_fwd: returns (dq1, dq2, dk, dv)."""
    _require_gpu(q1, q2, k, v, do1, do2)
    q1, q2, k, v, do1, do2, s, km = _aligned(q1, q2, k, v, do1, do2, s, km)
    L = lib()
    B, H, T, DK = q1.shape
    DV = v.shape[-1]
    code = dtype_code(q1)
    dev = q1.device
    dq1, dq2, dk, dv = torch.empty_like(q1), torch.empty_like(q2), torch.empty_like(k), torch.empty_like(v)
    with _on(dev):
        ws = _workspace(L.fbla_la_pair_workspace_bytes(1, B, H, T, DK, DV, code), dev)
        rc = L.fbla_la_pair_bwd(_ptr(q1), _ptr(q2), _ptr(k), _ptr(v), _ptr(do1), _ptr(do2), _ptr(s), _ptr(km),
                                _ptr(dq1), _ptr(dq2), _ptr(dk), _ptr(dv), _ptr(ws), ws.numel(), B, H, T, DK, DV,
                                code, float(scale), float(eps), _stream(dev))
    _check(rc, "fbla_la_pair_bwd")
    return dq1, dq2, dk, dv


def varlen_fwd(q, k, v, cu_seqlens, max_seqlen, scale, eps, extra_flags=0):
    """Packed forward: returns (o, s, km).  Tensors contiguous [T,H,D]."""
    _require_gpu(q, k, v, cu_seqlens)
    q, k, v, cu_seqlens = _aligned(q, k, v, cu_seqlens)
    L = lib()
    T, H, DK = q.shape
    DV = v.shape[-1]
    N = cu_seqlens.numel() - 1
    code = dtype_code(q)
    dev = q.device
    flags = NORMALIZE | (DEFAULT_SCALE if scale is None else 0) | extra_flags
    o = torch.empty_like(v)
    s = torch.empty(N, H, DK, DV, dtype=torch.float32, device=dev)
    km = torch.empty(N, H, DK, dtype=torch.float32, device=dev)
    with _on(dev):
        ws = _workspace(L.fbla_varlen_workspace_bytes(0, T, N, H, max_seqlen, DK, DV, code, flags), dev)
        rc = L.fbla_varlen_fwd(_ptr(q), _ptr(k), _ptr(v), _ptr(cu_seqlens), _ptr(o), _ptr(s),
                               _ptr(km), _ptr(ws), ws.numel(), T, N, H, max_seqlen, DK, DV, code,
                               flags, 0.0 if scale is None else float(scale), float(eps),
                               _stream(dev))
    _check(rc, "fbla_varlen_fwd")
    return o, s, km


def varlen_bwd(q, k, v, cu_seqlens, max_seqlen, do, s, km, scale, eps, extra_flags=0):
    """Packed backward: returns (dq, dk, dv)."""
    _require_gpu(q, k, v, do, cu_seqlens)
    q, k, v, do, cu_seqlens, s, km = _aligned(q, k, v, do, cu_seqlens, s, km)
    L = lib()
    T, H, DK = q.shape
    DV = v.shape[-1]
    N = cu_seqlens.numel() - 1
    code = dtype_code(q)
    dev = q.device
    flags = NORMALIZE | (DEFAULT_SCALE if scale is None else 0) | extra_flags
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    with _on(dev):
        ws = _workspace(L.fbla_varlen_workspace_bytes(1, T, N, H, max_seqlen, DK, DV, code, flags), dev)
        rc = L.fbla_varlen_bwd(_ptr(q), _ptr(k), _ptr(v), _ptr(cu_seqlens), _ptr(do), _ptr(s),
                               _ptr(km), _ptr(dq), _ptr(dk), _ptr(dv), _ptr(ws), ws.numel(), T, N,
                               H, max_seqlen, DK, DV, code, flags,
                               0.0 if scale is None else float(scale), float(eps), _stream(dev))
    _check(rc, "fbla_varlen_bwd")
    return dq, dk, dv


def chunk_reduce(q, k, v, chunk, with_norm=False, p_norm=2.0):
    """Block statistics of piecewise attention.  q,k:[B,H,T,K] v:[B,H,T,V] contiguous.
    Returns fp32 (qc, kc, vc, h, h_norm or None)."""
    _require_gpu(q, k, v)
    q, k, v = _aligned(q, k, v)
    L = lib()
    B, H, T, K = k.shape
    V = v.shape[-1]
    NT = -(-T // chunk)
    code = dtype_code(q)
    dev = q.device
    f32 = dict(dtype=torch.float32, device=dev)
    qc, kc = torch.empty(B, H, NT, K, **f32), torch.empty(B, H, NT, K, **f32)
    vc, h = torch.empty(B, H, NT, V, **f32), torch.empty(B, H, K, V, **f32)
    h_norm = torch.empty(B, H, NT, **f32) if with_norm else None
    with _on(dev):
        ws = _workspace(L.fbla_chunk_reduce_workspace_bytes(B * H, T, K, V, chunk, code, int(with_norm)), dev)
        rc = L.fbla_chunk_reduce(_ptr(q), _ptr(k), _ptr(v), _ptr(qc), _ptr(kc), _ptr(vc), _ptr(h),
                                 _ptr(h_norm), _ptr(ws), ws.numel(), B * H, T, K, V, chunk,
                                 float(p_norm), code, _stream(dev))
    _check(rc, "fbla_chunk_reduce")
    return qc, kc, vc, h, h_norm


def select_blocks(qc, kc, bias, top_k, scale):
    """Indices (int32, ascending) of the top_k key blocks per query block; qc, kc fp32 [B,H,NT,K]."""
    _require_gpu(qc, kc, bias)
    qc, kc, bias = _aligned(qc, kc, bias)
    L = lib()
    B, H, NT, K = qc.shape
    dev = qc.device
    idx = torch.empty(B, H, NT, top_k, dtype=torch.int32, device=dev)
    with _on(dev):
        rc = L.fbla_select_blocks(_ptr(qc), _ptr(kc), _ptr(bias), _ptr(idx), B * H, NT, K, top_k,
                                  float(scale), _stream(dev))
    _check(rc, "fbla_select_blocks")
    return idx


def piecewise_supported(q, v, block):
    B, H, T, K = q.shape
    return bool(q.dtype in _DTYPES and
                lib().fbla_piecewise_workspace_bytes(B * H, T, K, v.shape[-1], block, dtype_code(q)))


def piecewise_fwd(q, k, v, kc, vc, h, indices, block, scale):
    """Piecewise attention forward; indices int32 [B,H,NT,NS]; kc, vc, h fp32 from chunk_reduce."""
    _require_gpu(q, k, v, kc, vc, h, indices)
    q, k, v, kc, vc, h, indices = _aligned(q, k, v, kc, vc, h, indices)
    L = lib()
    B, H, T, K = q.shape
    V = v.shape[-1]
    NS = indices.shape[-1]
    code = dtype_code(q)
    dev = q.device
    o = torch.empty_like(v)
    with _on(dev):
        ws = _workspace(L.fbla_piecewise_workspace_bytes(B * H, T, K, V, block, code), dev)
        rc = L.fbla_piecewise_fwd(_ptr(q), _ptr(k), _ptr(v), _ptr(kc), _ptr(vc), _ptr(h), _ptr(indices),
                                  _ptr(o), _ptr(ws), ws.numel(), B * H, T, K, V, block, NS,
                                  float(scale), code, _stream(dev))
    _check(rc, "fbla_piecewise_fwd")
    return o


def elu1_fwd(x0, x1=None):
    """elu(x) + 1 of one or two contiguous tensors in one launch: returns the new tensor(s)."""
    _require_gpu(x0, x1)
    x0, x1 = _aligned(x0, x1)
    L = lib()
    y0 = torch.empty_like(x0)
    y1 = torch.empty_like(x1) if x1 is not None else None
    if x1 is not None and (x1.dtype != x0.dtype or x1.device != x0.device):
        raise ValueError("elu1_fwd: both tensors must have the same dtype and device")
    with _on(x0.device):
        rc = L.fbla_elu1_fwd(_ptr(x0), _ptr(y0), x0.numel(), _ptr(x1), _ptr(y1),
                             x1.numel() if x1 is not None else 0, dtype_code(x0), _stream(x0.device))
    _check(rc, "fbla_elu1_fwd")
    return y0 if x1 is None else (y0, y1)


def elu1_bwd(x, dy):
    """dy * d(elu(x) + 1)/dx for contiguous tensors of the same shape and dtype."""
    _require_gpu(x, dy)
    x, dy = _aligned(x, dy)
    L = lib()
    dx = torch.empty_like(x)
    with _on(x.device):
        rc = L.fbla_elu1_bwd(_ptr(x), _ptr(dy), _ptr(dx), x.numel(), dtype_code(x), _stream(x.device))
    _check(rc, "fbla_elu1_bwd")
    return dx


def _rows(t):
    """(tensor, batch stride, row stride) of token rows [B, N, C] the depth-wise kernels can read in place: channels
    adjacent, rows and batches at whole 16-byte pieces; anything else is copied to contiguous memory."""
    piece = 16 // t.element_size()
    if t.stride(2) != 1 or t.stride(0) % piece or t.stride(1) % piece or t.stride(1) < t.shape[2] or \
            t.stride(0) < t.shape[2] or t.data_ptr() % 16:
        t = t.clone(memory_format=torch.contiguous_format)
    return t, t.stride(0), t.stride(1)


def dwconv_fwd(x, w, bias, H, W, flip=False):
    """Depth-wise convolution of token rows x [B, H*W, C] with w [Cw, 1, K, K]; returns contiguous [B, H*W, C]."""
    B, N, C = x.shape
    if N != H * W or H < 1:
        raise ValueError(f"dwconv_fwd: x must be rows of H * W tokens, got {tuple(x.shape)} for H = {H}, W = {W}")
    if w.dtype != x.dtype or (bias is not None and bias.dtype != x.dtype):
        raise ValueError("dwconv_fwd: x, w and bias must have one dtype")
    _require_gpu(x, w, bias)
    x, x_batch, x_row = _rows(x)
    y = torch.empty(B, N, C, dtype=x.dtype, device=x.device)
    with _on(x.device):
        rc = lib().fbla_dwconv_fwd(_ptr(x), x_batch, x_row, _ptr(w), _ptr(bias), _ptr(y), N * C, C, B, H, W, C,
                                   w.shape[0], w.shape[-1], int(flip), dtype_code(x), _stream(x.device))
    _check(rc, "fbla_dwconv_fwd")
    return y


def dwconv_grad(x, g, w, H, W, with_bias):
    """(dw, db or None) of dwconv_fwd from its input and its output's gradient, both [B, H*W, C]."""
    B, N, C = x.shape
    if N != H * W or H < 1:
        raise ValueError(f"dwconv_grad: x must be rows of H * W tokens, got {tuple(x.shape)} for H = {H}, W = {W}")
    if g.shape != x.shape:
        raise ValueError(f"dwconv_grad: x and g must have one shape, got {tuple(x.shape)} and {tuple(g.shape)}")
    if w.dtype != x.dtype or g.dtype != x.dtype:
        raise ValueError("dwconv_grad: x, g and w must have one dtype")
    _require_gpu(x, g, w)
    x, x_batch, x_row = _rows(x)
    g, g_batch, g_row = _rows(g)
    Cw, K, code = w.shape[0], w.shape[-1], dtype_code(x)
    L = lib()
    dw = torch.empty_like(w, memory_format=torch.contiguous_format)
    db = torch.empty(Cw, dtype=w.dtype, device=w.device) if with_bias else None
    with _on(x.device):
        ws = _workspace(L.fbla_dwconv_grad_workspace_bytes(B, H, W, C, Cw, K, code), x.device)
        rc = L.fbla_dwconv_grad(_ptr(x), x_batch, x_row, _ptr(g), g_batch, g_row, _ptr(dw), _ptr(db), _ptr(ws),
                                ws.numel(), B, H, W, C, Cw, K, code, _stream(x.device))
    _check(rc, "fbla_dwconv_grad")
    return dw, db


def _token_rows(t):
    """(tensor, row stride) of t [..., C] as rows the projection kernels can read in place: channels adjacent, whole
    16-byte pieces between the rows; anything else is copied to contiguous memory."""
    rows = t.reshape(-1, t.shape[-1])
    if rows.stride(1) != 1 or rows.stride(0) * rows.element_size() % 16 or rows.stride(0) < rows.shape[1] or rows.data_ptr() % 16:
        rows = rows.clone(memory_format=torch.contiguous_format)
    return rows, rows.stride(0)


def linear_wgrad(g, x, with_bias):
    """(dw [M, N], db [M] or None) of y = x W^T + b from the output's gradient g [..., M] and x [..., N]."""
    _require_gpu(g, x)
    g, g_row = _token_rows(g)
    x, x_row = _token_rows(x)
    (T, M), N, code = g.shape, x.shape[1], dtype_code(x)
    if x.shape[0] != T or g.dtype != x.dtype or g.device != x.device:
        raise ValueError("linear_wgrad: g and x must agree in tokens, dtype and device")
    L, dev = lib(), x.device
    dw = torch.empty(M, N, dtype=x.dtype, device=dev)
    db = torch.empty(M, dtype=x.dtype, device=dev) if with_bias else None
    with _on(dev):
        ws = _workspace(L.fbla_linear_wgrad_workspace_bytes(T, M, N, code), dev)
        rc = L.fbla_linear_wgrad(_ptr(g), g_row, _ptr(x), x_row, _ptr(dw), _ptr(db), _ptr(ws), ws.numel(), T, M, N,
                                 code, _stream(dev))
    _check(rc, "fbla_linear_wgrad")
    return dw, db


def _whole(*tensors):
    """The tensors in contiguous, 16-byte aligned memory (copies where they are not)."""
    return _aligned(*(t if t is None else t.contiguous() for t in tensors))


def polarity_fwd(qg, kv, pe, scale, power, heads):
    """Polarity features of qg [B, N, 2C] and kv [B, n, 2C]: (q_same, q_opp [B, heads, N, 2d], k_both [B, heads, n, 2d],
    v [B, heads, n, d]).  pe [1, n, C], scale [1, 1, C], power [1, heads, 1, d]."""
    _require_gpu(qg, kv, pe, scale, power)
    qg, kv, pe, scale, power = _whole(qg, kv, pe, scale, power)
    B, N, C2 = qg.shape
    n, d = kv.shape[1], C2 // 2 // heads
    q_same = torch.empty(B, heads, N, 2 * d, dtype=qg.dtype, device=qg.device)
    q_opp = torch.empty_like(q_same)
    k_both = torch.empty(B, heads, n, 2 * d, dtype=qg.dtype, device=qg.device)
    v = torch.empty(B, heads, n, d, dtype=qg.dtype, device=qg.device)
    with _on(qg.device):
        rc = lib().fbla_polarity_fwd(_ptr(qg), _ptr(kv), _ptr(pe), _ptr(scale), _ptr(power), _ptr(q_same), _ptr(q_opp),
                                     _ptr(k_both), _ptr(v), B, N, n, heads, d, dtype_code(qg), _stream(qg.device))
    _check(rc, "fbla_polarity_fwd")
    return q_same, q_opp, k_both, v


def polarity_bwd(qg, kv, pe, scale, power, heads, dq_same, dq_opp, dk_both, dv, dv_rows, dgate):
    """Gradients (dqg, dkv, dpe, dscale, dpower) of polarity_fwd; dv_rows [B, n, C] and dgate [B, N, C] are the gradients of
    kv's and qg's second halves as rows."""
    tensors = qg, kv, pe, scale, power, dq_same, dq_opp, dk_both, dv, dv_rows, dgate
    _require_gpu(*tensors)
    tensors = _whole(*tensors)
    qg, kv, pe, scale, power = tensors[:5]
    B, N, C2 = qg.shape
    n, d, code, L = kv.shape[1], C2 // 2 // heads, dtype_code(qg), lib()
    grads = tuple(torch.empty_like(t) for t in tensors[:5])
    with _on(qg.device):
        ws = _workspace(L.fbla_polarity_bwd_workspace_bytes(B, N, n, heads, d, code), qg.device)
        rc = L.fbla_polarity_bwd(*(_ptr(t) for t in tensors + grads), _ptr(ws), ws.numel(), B, N, n, heads, d, code,
                                 _stream(qg.device))
    _check(rc, "fbla_polarity_bwd")
    return grads


def rotary_fwd(qk, x, rotations, heads):
    """Rotary features of qk [B, N, 2C] and the values x [B, N, C]: (q, k, q_rot, k_rot, v) [B, heads, N, d]; rotations
    fp32 [..., pairs, 2] over the N tokens."""
    _require_gpu(qk, x, rotations)
    qk, x, rotations = _whole(qk, x, rotations)
    B, N, C = x.shape
    out = tuple(torch.empty(B, heads, N, C // heads, dtype=x.dtype, device=x.device) for _ in range(5))
    with _on(x.device):
        rc = lib().fbla_rotary_fwd(_ptr(qk), _ptr(x), _ptr(rotations), 2 * rotations.shape[-2], *(_ptr(t) for t in out), B, N,
                                   heads, C // heads, dtype_code(x), _stream(x.device))
    _check(rc, "fbla_rotary_fwd")
    return out


def rotary_bwd(qk, rotations, heads, dq, dk, dq_rot, dk_rot, dv, dv_rows):
    """Gradients (dqk, dx) of rotary_fwd; dv_rows [B, N, C] is added to the values' gradient."""
    tensors = qk, rotations, dq, dk, dq_rot, dk_rot, dv, dv_rows
    _require_gpu(*tensors)
    qk, rotations, *rest = _whole(*tensors)
    B, N, C = dv_rows.shape
    dqk, dx = torch.empty_like(qk), torch.empty_like(rest[-1])
    with _on(qk.device):
        rc = lib().fbla_rotary_bwd(_ptr(qk), _ptr(rotations), 2 * rotations.shape[-2], *(_ptr(t) for t in rest), _ptr(dqk),
                                   _ptr(dx), B, N, heads, C // heads, dtype_code(qk), _stream(qk.device))
    _check(rc, "fbla_rotary_bwd")
    return dqk, dx


def merge_fwd(o, o2, local, gate):
    """(heads + local) * gate as rows [B, N, C]: o [B, heads, N, d], or o and o2 [B, heads, N, d / 2] each; gate or None."""
    _require_gpu(o, o2, local, gate)
    o, o2, local = _whole(o, o2, local)
    gate, _, gate_row = _rows_of_batches(gate)
    B, heads, N, d = o.shape
    d = d if o2 is None else 2 * d
    out = torch.empty_like(local)
    with _on(o.device):
        rc = lib().fbla_merge_fwd(_ptr(o), _ptr(o2), _ptr(local), _ptr(gate), gate_row, _ptr(out), B, N, heads, d,
                                  dtype_code(o), _stream(o.device))
    _check(rc, "fbla_merge_fwd")
    return out


def merge_bwd(dout, heads, halves, o, o2, local, gate):
    """Gradients (do, do2 or None, dlocal, dgate or None) of merge_fwd; without a gate o, o2 and local are not looked at."""
    _require_gpu(dout, o, o2, local, gate)
    dout, o, o2, local = _whole(dout, o, o2, local)
    gate, _, gate_row = _rows_of_batches(gate)
    B, N, C = dout.shape
    d = C // heads
    d_o = torch.empty(B, heads, N, d // 2 if halves else d, dtype=dout.dtype, device=dout.device)
    d_o2 = torch.empty_like(d_o) if halves else None
    dlocal, dgate = (torch.empty_like(dout), torch.empty_like(dout)) if gate is not None else (dout, None)
    with _on(dout.device):
        rc = lib().fbla_merge_bwd(_ptr(dout), _ptr(o), _ptr(o2), _ptr(local), _ptr(gate), gate_row, _ptr(d_o), _ptr(d_o2),
                                  _ptr(dlocal) if gate is not None else None, _ptr(dgate), B, N, heads, d, dtype_code(dout),
                                  _stream(dout.device))
    _check(rc, "fbla_merge_bwd")
    return d_o, d_o2, dlocal, dgate


def _rows_of_batches(t):
    """As _rows, for rows that lie at one distance over all batches; None stays None."""
    if t is None:
        return None, 0, 0
    t, batch, row = _rows(t)
    if batch != row * t.shape[1]:
        t = t.clone(memory_format=torch.contiguous_format)
    return t, t.stride(0), t.stride(1)


def interpolate_fwd(x, tokens):
    """Token rows x [B, n, C] linearly interpolated to [B, tokens, C]."""
    _require_gpu(x)
    x, x_batch, x_row = _rows(x)
    B, n, C = x.shape
    y = torch.empty(B, tokens, C, dtype=x.dtype, device=x.device)
    with _on(x.device):
        rc = lib().fbla_interpolate_fwd(_ptr(x), x_batch, x_row, _ptr(y), B, n, tokens, C, dtype_code(x), _stream(x.device))
    _check(rc, "fbla_interpolate_fwd")
    return y


def interpolate_bwd(g, n):
    """Gradient [B, n, C] of interpolate_fwd from the output's gradient g [B, tokens, C]."""
    _require_gpu(g)
    g, = _whole(g)
    B, tokens, C = g.shape
    dx = torch.empty(B, n, C, dtype=g.dtype, device=g.device)
    with _on(g.device):
        rc = lib().fbla_interpolate_bwd(_ptr(g), _ptr(dx), B, n, tokens, C, dtype_code(g), _stream(g.device))
    _check(rc, "fbla_interpolate_bwd")
    return dx


def focus_fwd(q, kv, pe, scale, heads):
    """Focused features of q [B, N, C] and kv [B, n, 2C]: (q, k, v) as [B, heads, tokens, d]."""
    _require_gpu(q, kv, pe, scale)
    q, kv, pe, scale = _whole(q, kv, pe, scale)
    B, N, C = q.shape
    n = kv.shape[1]
    out = tuple(torch.empty(B, heads, t, C // heads, dtype=q.dtype, device=q.device) for t in (N, n, n))
    with _on(q.device):
        rc = lib().fbla_focus_fwd(_ptr(q), _ptr(kv), _ptr(pe), _ptr(scale), *(_ptr(t) for t in out), B, N, n, heads,
                                  C // heads, dtype_code(q), _stream(q.device))
    _check(rc, "fbla_focus_fwd")
    return out


def focus_bwd(q, kv, pe, scale, heads, dq_heads, dk_heads, dv_heads, dv_rows):
    """Gradients (dq, dkv, dpe, dscale) of focus_fwd; dv_rows [B, n, C] is added to the values' gradient."""
    tensors = q, kv, pe, scale, dq_heads, dk_heads, dv_heads, dv_rows
    _require_gpu(*tensors)
    tensors = _whole(*tensors)
    q, kv = tensors[:2]
    (B, N, C), n, code, L = q.shape, kv.shape[1], dtype_code(q), lib()
    grads = tuple(torch.empty_like(t) for t in tensors[:4])
    with _on(q.device):
        ws = _workspace(L.fbla_focus_bwd_workspace_bytes(B, N, n, heads, C // heads, code), q.device)
        rc = L.fbla_focus_bwd(*(_ptr(t) for t in tensors + grads), _ptr(ws), ws.numel(), B, N, n, heads, C // heads, code,
                              _stream(q.device))
    _check(rc, "fbla_focus_bwd")
    return grads


def most_row_channels(t):
    """The widest row of t's type that focus_fwd takes."""
    return 4096 // t.element_size()


def turn_fwd(q, k, weight, rotations):
    """(k * weight, q turned, k * weight turned) of heads [B, heads, N, d]; weight [B, heads, N, 1], rotations fp32
    [..., d / 2, 2] over the N tokens."""
    _require_gpu(q, k, weight, rotations)
    q, k, weight, rotations = _whole(q, k, weight, rotations)
    B, heads, N, d = q.shape
    out = tuple(torch.empty_like(q) for _ in range(3))
    with _on(q.device):
        rc = lib().fbla_turn_fwd(_ptr(q), _ptr(k), _ptr(weight), _ptr(rotations), *(_ptr(t) for t in out), B, N, heads, d,
                                 dtype_code(q), _stream(q.device))
    _check(rc, "fbla_turn_fwd")
    return out


def turn_bwd(k, weight, rotations, dk_out, dq_rot, dk_rot):
    """Gradients (dq, dk, dweight) of turn_fwd."""
    tensors = k, weight, rotations, dk_out, dq_rot, dk_rot
    _require_gpu(*tensors)
    tensors = _whole(*tensors)
    k, weight = tensors[:2]
    B, heads, N, d = k.shape
    grads = torch.empty_like(k), torch.empty_like(k), torch.empty_like(weight)
    with _on(k.device):
        rc = lib().fbla_turn_bwd(*(_ptr(t) for t in tensors + grads), B, N, heads, d, dtype_code(k), _stream(k.device))
    _check(rc, "fbla_turn_bwd")
    return grads
