"""The calls of pyext/calls.cpp through ctypes, for a Python or torch that the extension module
was not built for (it is bound to one of each; libmbrt.so is not).  Same functions, arguments,
checks and errors; a call takes about 5 us more of host time.
"""
from __future__ import annotations

import ctypes as C

import torch

from . import _abi

_DT = {torch.float32: _abi.F32, torch.float16: _abi.F16, torch.int64: _abi.I64, torch.bfloat16: _abi.BF16,
       torch.int32: _abi.I32}


def _tensors(*ts):
    for t in ts:
        if not isinstance(t, torch.Tensor):
            raise TypeError("mbrt: expected a torch.Tensor")


def _contig(*ts):
    _tensors(*(t for t in ts if t is not None))
    for t in ts:
        if t is not None and not t.is_contiguous():
            raise ValueError("mbrt: expected a contiguous tensor")


def _dt(t, none=None):
    if t is None:
        return none
    try:
        return _DT[t.dtype]
    except KeyError as e:
        raise TypeError(f"mbrt: unsupported dtype {t.dtype}") from e


def _p(t):
    return C.c_void_p(0 if t is None else t.data_ptr())


def _s(stream):
    return C.c_void_p(torch.cuda.current_stream().cuda_stream if stream is None else stream)


def _float(x):
    return C.c_double(x).value  # a number as the C-ABI takes it: no text


def fill(t, value, stream):
    _tensors(t)
    _contig(t)
    _abi.call("mbrt_fill", _p(t), _dt(t), t.numel(), _float(value), _s(stream))


def strided_copy(src, dst, stream):
    _tensors(src, dst)
    _contig(dst)
    if src.shape != dst.shape:
        raise ValueError("strided_copy: shape mismatch")
    m = _abi.StridedMeta()
    m.ndim = src.dim()
    for d in range(src.dim()):
        m.dst_shape[d] = src.shape[d]
        m.src_strides[d] = src.stride(d)
    _abi.call("mbrt_strided_copy", _p(src), _p(dst), _dt(src), C.byref(m), _s(stream))


def pad(src, out, before, value, reflect, stream):
    _tensors(src, out)
    _contig(src, out)
    m = _abi.PadMeta()
    m.ndim = src.dim()
    for d in range(src.dim()):
        m.src_shape[d] = src.shape[d]
        m.dst_shape[d] = out.shape[d]
        m.pad_before[d] = before[d]
    if reflect:
        _abi.call("mbrt_pad_reflect", _p(src), _p(out), _dt(src), C.byref(m), _s(stream))
    else:
        _abi.call("mbrt_pad_const", _p(src), _p(out), _dt(src), C.byref(m), _float(value), _s(stream))


def cat(srcs, dim, out, stream):
    srcs = list(srcs)
    _tensors(out, *srcs)
    _contig(out, *srcs)
    dim = dim % out.dim()
    outer = inner = 1
    for d in range(dim):
        outer *= out.shape[d]
    for d in range(dim + 1, out.dim()):
        inner *= out.shape[d]
    arr = (_abi.CatSrc * len(srcs))()
    off = 0
    for i, s in enumerate(srcs):
        arr[i].ptr = s.data_ptr()
        arr[i].dim_size = s.shape[dim]
        arr[i].dim_offset = off
        off += s.shape[dim]
    _abi.call("mbrt_cat", _p(out), arr, len(srcs), outer, out.shape[dim], inner * out.element_size(), _s(stream))


def rms_norm(x, gamma, out, scale, eps, stream):
    _tensors(x, gamma, out)
    _contig(x, gamma, out)
    dim = x.shape[-1]
    _abi.call("mbrt_rms_norm", _p(x), _dt(x), _p(gamma), _dt(gamma), _p(out), _dt(out), x.numel() // dim, dim,
              _float(scale), _float(eps), _s(stream))


def residual_add_rms_norm(residual, update, gamma, sum_out, normed, scale, eps, stream):
    _tensors(residual, update, gamma, normed)
    _contig(residual, update, gamma, sum_out, normed)
    dim = residual.shape[-1]
    _abi.call("mbrt_residual_add_rms_norm", _p(residual), _p(update), _dt(residual), _p(gamma), _dt(gamma), _p(sum_out),
              _dt(sum_out, _dt(residual)), _p(normed), _dt(normed), residual.numel() // dim, dim, _float(scale),
              _float(eps), _s(stream))


def bias_act(x, bias, out, act, stream):
    _tensors(x, out)
    _contig(x, bias, out)
    cols = x.shape[-1]
    _abi.call("mbrt_bias_act", _p(x), _dt(x), _p(bias), _dt(bias, _abi.F32), _p(out), _dt(out), x.numel() // cols, cols,
              act, _s(stream))


def glu(x, out, stream):
    _tensors(x, out)
    _contig(x, out)
    full = x.shape[-1]
    if full % 2:
        raise ValueError("glu_last_dim: last dimension must be even")
    _abi.call("mbrt_glu_last_dim", _p(x), _dt(x), _p(out), _dt(out), x.numel() // full, full // 2, _s(stream))


def gate_merge(attn, gate, out, layout, gate_is_logit, stream):
    _tensors(attn, gate, out)
    _contig(attn, gate, out)
    if attn.dim() != 4:
        raise ValueError("gate_merge: expected a 4-d attention output")
    if layout == _abi.LAYOUT_BHND:
        B, H, N, D = attn.shape
    else:
        B, N, H, D = attn.shape
    _abi.call("mbrt_sigmoid_gate_merge", _p(attn), _dt(attn), _p(gate), _dt(gate), int(bool(gate_is_logit)), _p(out),
              _dt(out), B, H, N, D, layout, _s(stream))


def softmax(x, out, scale, stream):
    _tensors(x, out)
    _contig(x, out)
    cols = x.shape[-1]
    _abi.call("mbrt_softmax_rows", _p(x), _dt(x), _p(out), _dt(out), x.numel() // cols, cols, _float(scale), _s(stream))


def split_qkv_rotary(qkv, cos, sin, q, k, v, heads, stream):
    _tensors(qkv, cos, sin, q, k, v)
    _contig(qkv, cos, sin, q, k, v)
    if qkv.dim() != 3:
        raise ValueError("split_qkv_rotary: expected qkv [B, N, 3 H D]")
    B, N, three_hd = qkv.shape
    _abi.call("mbrt_split_qkv_heads_rotary", _p(qkv), _dt(qkv), _p(cos), _p(sin), _dt(cos), _p(q), _p(k), _p(v), _dt(q),
              B, N, heads, three_hd // (3 * heads), q.shape[2], _s(stream))


def attention_ex(q, k, v, sizes, strides, cos, sin, gate, gate_is_logit, out, scale, p_precision, stream):
    _tensors(q, k, v, out, *(t for t in (cos, sin, gate) if t is not None))
    _abi.call("mbrt_attention_ex", _p(q), _p(k), _p(v), _dt(q), *sizes, *strides, _p(cos), _p(sin), _dt(cos, _abi.F32),
              _p(gate), _dt(gate, _abi.F32), int(bool(gate_is_logit)), _p(out), _dt(out), _float(scale), p_precision,
              _s(stream))


def stft(x, window, hop, center, normalized, out, n_fft, win_length, stream):
    _tensors(x, window, out)
    _contig(x, window, out)
    _abi.call("mbrt_stft", _p(x), _p(window), _p(out), x.shape[0], x.shape[1], n_fft, hop, win_length, window.numel(),
              int(bool(center)), int(bool(normalized)), _s(stream))


def istft(spec, window, hop, center, normalized, length, out, workspace, n_fft, win_length, stream):
    _tensors(spec, window, out, workspace)
    _contig(spec, window, out)
    if spec.dim() != 4:
        raise ValueError("istft: expected a spectrum [B, F, T, 2]")
    B, F, T, _ = spec.shape
    _abi.call("mbrt_istft", _p(spec), _dt(spec), _p(window), _p(out), B, F, T, n_fft, hop, win_length, window.numel(),
              int(bool(center)), int(bool(normalized)), length, _p(workspace),
              workspace.numel() * workspace.element_size(), _s(stream))


def chunk_accumulate(dest, weight_sum, src, window, offset, stream):
    _tensors(dest, weight_sum, src, window)
    _contig(dest, weight_sum, src, window)
    n = src.shape[-1]
    _abi.call("mbrt_chunk_accumulate", _p(dest), _p(weight_sum), _p(src), _p(window), src.numel() // max(n, 1), n,
              dest.shape[-1], offset, _s(stream))
