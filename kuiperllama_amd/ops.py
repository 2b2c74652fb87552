"""Operator-level Python mirror of the reference's kernel interface
(kuiper/source/op/kernels/kernels_interface.h:6-68) over libkuiper_hip.so.

Arguments are torch tensors living on the GPU (torch is only the owner of device memory and
streams here); every call goes through the C-ABI and launches a hand-written HIP kernel on
torch's current stream.  There is no eager/CPU fallback: a CPU tensor is an error.
"""
from __future__ import annotations

import os
from typing import Optional

import torch

from . import _ffi

ROPE_INTERLEAVED, ROPE_HALF = 0, 1


def _p(t: Optional[torch.Tensor], dtype=None):
    if t is None:
        return None
    if not t.is_cuda:
        raise ValueError("kuiperllama_amd.ops: tensors must be on the GPU (no CPU fallback)")
    if not t.is_contiguous():
        raise ValueError("kuiperllama_amd.ops: tensors must be contiguous")
    if dtype is not None and t.dtype != dtype:
        raise TypeError(f"expected {dtype}, got {t.dtype}")
    return t.data_ptr()


# The handle without building a torch.cuda.Stream for it: 2.5 of the 7.5 us that one
# operator call took on the host.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream():
    if _raw_stream is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(torch.cuda.current_device())


class _Unbound:
    """Stands for csrc/kh_pyops.c, the calls that a decoder layer is made of, until the first of them loads it."""

    def __getattr__(self, name):
        global _n
        import ctypes as C
        import importlib.machinery
        import importlib.util
        from .build import PYOPS_PATH as path
        L = _ffi.lib()
        if not os.path.exists(path):
            raise ImportError(f"{path} is missing: build it with `python -m kuiperllama_amd.build`, which needs this "
                              "interpreter's headers")
        spec = importlib.util.spec_from_loader("kh_pyops", importlib.machinery.ExtensionFileLoader("kh_pyops", path))
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        mod.bind(tuple(C.cast(f, C.c_void_p).value for f in (L.kh_add_f32, L.kh_swiglu_f32, L.kh_matmul_f32, L.kh_matmul_q8,
                                                             L.kh_rmsnorm_f32, L.kh_rope_f32, L.kh_mha_f32)),
                 (torch.float32, torch.int32, torch.int8, torch.Tensor, getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device),
                  _raw_stream, _stream, _ffi.check, C.ArgumentError))
        _n = mod
        return getattr(mod, name)


_n = _Unbound()


def add(in1, in2, out):
    return _n.add(in1, in2, out)


def matmul(x, w, out, scale: float = 1.0):
    return _n.matmul(x, w, out, scale)


def matmul_q8(x, w8, scales, group_size: int, out):
    return _n.matmul_q8(x, w8, scales, group_size, out)


def embedding(tokens, w, out):
    V, dim = w.shape
    _ffi.check(_ffi.lib().kh_embedding_f32(_p(tokens, torch.int32), tokens.numel(),
                                           _p(w, torch.float32), _p(out, torch.float32), dim, V,
                                           _stream()), "kh_embedding_f32")
    return out


def embedding_host_tokens(tokens, w, out):
    """EmbeddingKernel as the reference calls it: `tokens` is a HOST int32 array (numpy); the ids
    travel in the kernel arguments, up to 512 per launch (kh_embedding_f32_host)."""
    import numpy as np
    t = np.ascontiguousarray(tokens, dtype=np.int32)
    _ffi.check(_ffi.lib().kh_embedding_f32_host(t.ctypes.data, t.size, _p(w), _p(out), w.shape[1],
                                                w.shape[0], _stream()), "kh_embedding_f32_host")


def swiglu(a, b, out):
    return _n.swiglu(a, b, out)


def rmsnorm(x, w, out, eps: float):
    return _n.rmsnorm(x, w, out, eps)


def rope(q, k, pos, sin_cache, cos_cache, head_size: int, mode: int):
    """pos: python int, or a 1-element int32 GPU tensor (graph-capturable form)."""
    _n.rope(q, k, pos, sin_cache, cos_cache, head_size, mode)
    return q, k


def sincos_cache(head_size: int, seq_len: int, theta: float, sin_cache, cos_cache):
    _ffi.check(_ffi.lib().kh_sincos_cache_f32(head_size, seq_len, theta,
                                              _p(sin_cache, torch.float32),
                                              _p(cos_cache, torch.float32), _stream()),
               "kh_sincos_cache_f32")
    return sin_cache, cos_cache


def mha(pos, head_num, layer_index, seq_len, kv_dim, kv_mul, head_size, mha_out, q, score,
        kcache, vcache):
    return _n.mha(pos, head_num, layer_index, seq_len, kv_dim, kv_mul, head_size, mha_out, q, score, kcache, vcache)


def mha_prefill(pos0, n_tokens, head_num, layer_index, seq_len, kv_dim, kv_mul, head_size, mha_out, q,
                kcache, vcache):
    """Causal attention of n_tokens consecutive queries (rows of q) on the matrix cores."""
    _ffi.sync_env()  # KH_PG_ATTN_QT
    _ffi.check(_ffi.lib().kh_mha_prefill_f32(
        int(pos0), int(n_tokens), head_num, layer_index, seq_len, kv_dim, kv_mul, head_size,
        _p(mha_out, torch.float32), _p(q, torch.float32), _p(kcache, torch.float32),
        _p(vcache, torch.float32), _stream()), "kh_mha_prefill_f32")
    return mha_out


def mha_decode_workspace(head_num: int, head_size: int, seq_len: int, device):
    """Zeroed workspace tensor for mha_decode (None when no time split is needed)."""
    _ffi.sync_env()  # KH_ATTN_TLONG
    n = int(_ffi.lib().kh_mha_decode_workspace_bytes(head_num, head_size, seq_len))
    if n < 0:
        _ffi.check(n, "kh_mha_decode_workspace_bytes")
    return torch.zeros(n, dtype=torch.uint8, device=device) if n else None


def mha_decode(pos, head_num, layer_index, seq_len, kv_dim, kv_mul, head_size, mha_out, q, kcache,
               vcache, workspace):
    d_pos, ipos = (None, int(pos)) if not torch.is_tensor(pos) else (_p(pos, torch.int32), 0)
    _ffi.check(_ffi.lib().kh_mha_decode_f32(
        d_pos, ipos, head_num, layer_index, seq_len, kv_dim, kv_mul, head_size,
        _p(mha_out, torch.float32), _p(q, torch.float32), _p(kcache, torch.float32),
        _p(vcache, torch.float32), _p(workspace) if workspace is not None else None,
        workspace.numel() if workspace is not None else 0, _stream()), "kh_mha_decode_f32")
    return mha_out


def argmax(logits, out_index):
    _ffi.check(_ffi.lib().kh_argmax_f32(_p(logits, torch.float32), logits.numel(),
                                        _p(out_index, torch.int32), _stream()), "kh_argmax_f32")
    return out_index


def argmax_host(logits) -> int:
    import ctypes as C
    r = C.c_int64(-1)
    _ffi.check(_ffi.lib().kh_argmax_f32_host(_p(logits, torch.float32), logits.numel(),
                                             C.byref(r), _stream()), "kh_argmax_f32_host")
    return int(r.value)


def softmax_(x):
    _ffi.check(_ffi.lib().kh_softmax_f32(_p(x, torch.float32), x.numel(), _stream()),
               "kh_softmax_f32")
    return x


def scale_(scale: float, x):
    _ffi.check(_ffi.lib().kh_scale_f32(scale, _p(x, torch.float32), x.numel(), _stream()),
               "kh_scale_f32")
    return x


def scale_sum(value, scale, out, pos: int, size: int, stride: int):
    _ffi.check(_ffi.lib().kh_scale_sum_f32(_p(value, torch.float32), _p(scale, torch.float32),
                                           _p(out, torch.float32), pos, size, stride, _stream()),
               "kh_scale_sum_f32")
    return out
