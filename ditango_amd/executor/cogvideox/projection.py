"""q, k and v of the CogVideoX adapter in one launch (``dt_qkv_project``), where nothing but the arithmetic of its modules is to run."""
from __future__ import annotations

import torch
from torch.autograd import forward_ad
from torch.nn import LayerNorm, Linear, Parameter
from torch.nn.modules import module as _module

from ... import _hip
from ...producer import _f32

HEAD_DIM = 64
# Operations beyond which the library's products may be faster, the launches around them included (us, modules -> one launch): 48 heads x
# 2222 tokens x 3072 channels, 126 GFLOP, 153 -> 122; 3328 tokens, 188 GFLOP, 198 -> 173; 4454, 252 GFLOP, 239 -> 253; 8016 429 -> 458.
MOST_FLOPS = 2.0e11


_FORWARD = {Linear: Linear.forward, LayerNorm: LayerNorm.forward}   # (a tool may patch the class)


def _only_arithmetic() -> bool:
    """No mode, transform, autocast or forward-mode derivative that would see the modules' operations."""
    return not (torch._C._len_torch_function_stack() or torch._C._len_torch_dispatch_stack() or torch.is_autocast_enabled("cuda")
                or torch._C._functorch.peek_interpreter_stack() is not None or torch.compiler.is_compiling()
                or torch.jit.is_tracing() or _module._has_any_global_hook() or forward_ad._current_level >= 0)


def _plain(m, kind) -> bool:
    """A module of exactly this class, whose call is its forward."""
    return (type(m) is kind and "forward" not in m.__dict__ and kind.forward is _FORWARD[kind]
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks))


def _tokens(x) -> bool:
    return (type(x) is torch.Tensor and x.is_cuda and x.dim() == 3 and x.stride(2) == 1 and x.stride(0) % 8 == 0 and x.stride(1) % 8 == 0
            and x.data_ptr() % 16 == 0 and x.numel() > 0)


def _parameter(p, like, shape) -> bool:
    return (type(p) is Parameter or type(p) is torch.Tensor) and p.dtype is like.dtype and p.device == like.device and p.shape == shape \
        and p.is_contiguous() and p.data_ptr() % 16 == 0


def project_qkv(attn, text, video, rotary):
    """(q, k, v) ``[B,S,H,64]``, or None where the modules have to be called."""
    linears = (attn.to_q, attn.to_k, attn.to_v)
    if not (_only_arithmetic() and all(_plain(m, Linear) for m in linears) and _tokens(text) and _tokens(video)):
        return None
    if text.dtype is not video.dtype or video.dtype not in _hip.HALF_DTYPES or text.device != video.device or text.shape[0] != video.shape[0] \
            or text.shape[2] != video.shape[2]:
        return None
    heads, channels = attn.heads, video.shape[2]
    if 6.0 * video.shape[0] * (text.shape[1] + video.shape[1]) * heads * HEAD_DIM * channels > MOST_FLOPS:
        return None
    norms = (getattr(attn, "norm_q", None), getattr(attn, "norm_k", None))
    params = [p for m in linears for p in (m.weight, m.bias) if p is not None]
    if channels % 64 or not all(_parameter(m.weight, video, (heads * HEAD_DIM, channels)) for m in linears) \
            or not all(m.bias is None or _parameter(m.bias, video, (heads * HEAD_DIM,)) for m in linears) \
            or not all(n is None or (_plain(n, LayerNorm) and all(p is None or _parameter(p, video, (HEAD_DIM,)) for p in (n.weight, n.bias))) for n in norms):
        return None
    if torch.is_grad_enabled() and any(t.requires_grad for t in (text, video, *params)):
        return None
    cos = sin = None
    if rotary is not None:
        cos, sin = _f32(rotary[0], video.device), _f32(rotary[1], video.device)
        if cos.shape != (video.shape[1], HEAD_DIM) or sin.shape != cos.shape or cos.data_ptr() % 16 or sin.data_ptr() % 16:
            return None
    ropes = (rotary is not None, rotary is not None and not getattr(attn, "is_cross_attention", False))
    projections = []
    for m, norm, rope in zip(linears, (*norms, None), (*ropes, False)):
        if norm is None:
            projections.append((m.weight, m.bias, _hip.DT_NORM_NONE, None, None, 0.0, rope))
            continue
        projections.append((m.weight, m.bias, _hip.DT_NORM_LAYER, norm.weight, norm.bias, norm.eps, rope))
    return tuple(_hip.qkv_project(text, video, heads, projections, cos, sin))
