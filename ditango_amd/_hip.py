"""Binding of ``libditango_hip.so`` (the C ABI declared in ``include/ditango_hip.h``).

The launches of a layer call go through ``_ditango_host`` (``csrc/host_binding.cpp``), an extension module that checks
the tensors and fills the C ABI's argument tables; what runs once per generation goes through ctypes.  There is
no fallback: if a library has not been built, or an entry point returns an error code, the call raises.  PyTorch
only supplies device memory (``tensor.data_ptr()``) and the current stream.
"""
from __future__ import annotations

import ctypes
import importlib.util
import os
from pathlib import Path
from typing import List, Optional, Sequence, Tuple

import torch

LIB_PATH = Path(__file__).resolve().parent / "lib" / "libditango_hip.so"
HOST_PATH = LIB_PATH.parent / "_ditango_host.so"

DT_BF16, DT_FP32, DT_FP16 = 0, 1, 2
DT_LSE_BHS, DT_LSE_BSH = 0, 1
DT_NORM_NONE, DT_NORM_RMS, DT_NORM_LAYER = 0, 1, 2
DT_ROPE_NONE, DT_ROPE_INTERLEAVED, DT_ROPE_HALVES = 0, 1, 2
DT_ROUND_NORM_BF16, DT_ROUND_ROPE_BF16, DT_IO_FP16, DT_WEIGHTS_16 = 1, 2, 4, 8
DT_ATTN_Q_PRESCALED, DT_ATTN_FP16 = 1, 2
DT_MAX_CHUNKS = 40
DT_MAX_JOBS = 40
DT_MAX_JOB_ENTRIES = 64
DT_MAX_MERGE = 64
DT_MAX_SEGMENTS = 8
DT_NOALLOC_TAIL_SLOTS = 1024

c_i32, c_i64, c_f32, c_vp = ctypes.c_int32, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p
_P = ctypes.POINTER

_SIGNATURES = {
    "dt_version": (ctypes.c_int, []),
    "dt_last_error": (ctypes.c_char_p, []),
    "dt_attn_chunk_fwd": (ctypes.c_int, [c_vp, c_vp, c_vp, c_vp, c_vp, c_i32, c_i32, c_i32, c_i32, c_i32,
                                         c_i64, c_i64, c_i64, c_i64, c_i64, c_i64, c_f32, c_vp]),
    "dt_attn_chunk_f16_fwd": (ctypes.c_int, [c_vp, c_vp, c_vp, c_vp, c_vp, c_i32, c_i32, c_i32, c_i32, c_i32,
                                             c_i64, c_i64, c_i64, c_i64, c_i64, c_i64, c_f32, c_vp]),
    "dt_attn_chunk_f32_fwd": (ctypes.c_int, [c_vp, c_vp, c_vp, c_vp, c_vp, c_i32, c_i32, c_i32, c_i32, c_i32,
                                             c_i64, c_i64, c_i64, c_i64, c_i64, c_i64, c_f32, c_vp]),
    "dt_attn_jobs_f32_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                            c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), _P(c_i64), _P(c_i64),
                                            c_i32, _P(c_i32), _P(c_i32), _P(c_vp), _P(c_vp), c_f32, c_vp]),
    "dt_attn_jobs_f32_ws_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                               c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), _P(c_i64), _P(c_i64),
                                               c_i32, _P(c_i32), _P(c_i32), _P(c_vp), _P(c_vp), c_i32, c_f32, c_vp, c_i64, c_vp, c_i64,
                                               c_vp]),
    "dt_attn_jobs_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                        c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                        c_i32, _P(c_i32), _P(c_i32), _P(c_vp), _P(c_vp), c_f32, c_vp]),
    "dt_attn_seg_jobs_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                            c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                            c_i32, _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32),
                                            _P(c_vp), _P(c_vp), c_f32, c_vp]),
    "dt_attn_workspace_bytes": (ctypes.c_int64, []),
    "dt_attn_seg_jobs_ws_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                               c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                               c_i32, _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32),
                                               _P(c_vp), _P(c_vp), c_f32, c_i32, c_vp, c_i64, c_vp]),
    "dt_attn_seg_jobs_noalloc_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                                    c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                                    c_i32, _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32),
                                                    _P(c_vp), _P(c_vp), c_f32, c_i32, c_vp]),
    "dt_attn_merge_counters": (ctypes.c_int64, [c_i32, c_i32, c_i32]),
    "dt_attn_merges_in_launch": (ctypes.c_int, [c_i32] * 8),
    "dt_attn_jobs_merge_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                              c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                              c_i32, _P(c_i32), _P(c_i32), _P(c_vp), _P(c_vp), c_vp, c_f32, c_i32,
                                              c_vp, c_i64, c_vp]),
    "dt_attn_sched_merge_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                               c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                               c_vp, c_vp, c_i32, c_vp, c_i64, c_vp, c_i64, c_i32, c_vp, c_vp,
                                               c_vp, c_f32, c_i32, c_vp, c_i64, c_vp]),
    "dt_attn_sched_seg_ws_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                                c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                                c_vp, c_vp, c_i32, c_vp, c_i64, c_vp, c_i64, c_i32, c_vp, c_vp,
                                                c_i32, _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), c_f32, c_i32,
                                                c_vp, c_i64, c_vp]),
    "dt_attn_sched_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                         c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                         c_vp, c_vp, c_i32, c_vp, c_i64, c_vp, c_i64, c_i32, c_vp, c_vp,
                                         c_f32, c_vp]),
    "dt_attn_sched_seg_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                             c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                             c_vp, c_vp, c_i32, c_vp, c_i64, c_vp, c_i64, c_i32, c_vp, c_vp,
                                             c_i32, _P(c_i32), _P(c_i32), _P(c_i32), _P(c_i32), c_f32, c_vp]),
    "dt_attn_varlen_jobs_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                               c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                               c_i32, _P(c_i32), _P(c_i32), _P(c_i32), c_i32, c_vp, _P(c_vp), c_i32,
                                               _P(c_vp), _P(c_vp), c_f32, c_i32, c_vp]),
    "dt_attn_sched_varlen_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                                c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                                c_vp, c_vp, c_i32, c_vp, c_i64, c_vp, c_i64, c_i32, c_vp, c_vp,
                                                c_i32, c_vp, _P(c_vp), c_i32, c_f32, c_i32, c_vp]),
    "dt_attn_varlen_jobs_ws_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                               c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                               c_i32, _P(c_i32), _P(c_i32), _P(c_i32), c_i32, c_vp, _P(c_vp), c_i32,
                                               _P(c_vp), _P(c_vp), c_f32, c_i32, c_vp, c_i64, c_vp]),
    "dt_attn_sched_varlen_ws_fwd": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i64, c_i64, c_i64,
                                                c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i64), c_i64, c_i64,
                                                c_vp, c_vp, c_i32, c_vp, c_i64, c_vp, c_i64, c_i32, c_vp, c_vp,
                                                c_i32, c_vp, _P(c_vp), c_i32, c_f32, c_i32, c_vp, c_i64, c_vp]),
    "dt_zero_rows_from": (ctypes.c_int, [c_vp, c_i64, c_i64, c_vp, c_vp]),
    "dt_merge_states": (ctypes.c_int, [c_i32, _P(c_vp), _P(c_vp), _P(c_i32), _P(c_i32), c_vp, c_i32, c_vp, c_i32,
                                       c_i32, c_i32, c_i32, c_i32, c_vp]),
    "dt_cache_store": (ctypes.c_int, [c_vp, c_i32, c_vp, c_i32, c_vp, c_vp, c_i32, c_i32, c_i32, c_i32, c_vp]),
    "dt_cache_load": (ctypes.c_int, [c_vp, c_vp, c_vp, c_i32, c_vp, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp]),
    "dt_state_copy": (ctypes.c_int, [c_vp, c_i32, c_vp, c_i32, c_vp, c_i32, c_vp, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp]),
    "dt_build_schedule": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp, c_vp, c_vp, c_vp]),
    "dt_build_schedule_table": (ctypes.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_vp, c_vp, c_vp, c_vp]),
    "dt_rel_l1_sums": (ctypes.c_int, [c_vp, c_vp, c_i64, c_vp, c_vp]),
    "dt_qkv_project": (ctypes.c_int, [c_vp, c_i64, c_i64, c_i32, c_vp, c_i64, c_i64, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp, c_vp, c_vp,
                                      c_i32, c_vp]),
    "dt_qk_norm_rope": (ctypes.c_int, [c_vp, c_i64, c_i64, c_i64, c_vp, c_i32, c_i32, c_i32, c_i32,
                                       c_i32, c_vp, c_vp, c_f32, c_i32, c_vp, c_vp, c_i64, c_i32, c_i32,
                                       _P(c_i32), c_i32, c_i32, c_f32, c_vp]),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)

_lib: Optional[ctypes.CDLL] = None


class DitangoHipError(RuntimeError):
    pass


def load_library(path: Optional[os.PathLike] = None) -> ctypes.CDLL:
    """Load the built library (once) and declare the signatures.  Raises if it is absent."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    p = Path(path) if path is not None else LIB_PATH
    if not p.exists():
        raise DitangoHipError(
            f"{p} is missing: build it with `python -m ditango_amd.build` "
            "(there is no non-HIP fallback for this path)")
    lib = ctypes.CDLL(str(p))
    for name, (res, args) in _SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    if path is None:
        _lib = lib
    return lib


_host_module = None


def _host():
    """The extension module (loaded once; raises if it is absent)."""
    global _host_module
    if _host_module is None:
        if not HOST_PATH.exists():
            raise DitangoHipError(f"{HOST_PATH} is missing: build it with `python -m ditango_amd.build`")
        spec = importlib.util.spec_from_file_location("_ditango_host", HOST_PATH)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        module.set_error_class(DitangoHipError)
        _host_module = module
    return _host_module


def _check(rc: int, what: str) -> None:
    if rc != 0:
        msg = load_library().dt_last_error().decode("utf-8", "replace")
        raise DitangoHipError(f"{what} failed with code {rc}: {msg}")


_raw_stream = torch._C._cuda_getCurrentRawStream   # device index -> handle of its current stream, without building a Stream
_current_device = torch._C._cuda_getDevice


def _stream() -> int:
    return _raw_stream(_current_device())


def _dtype_code(t: torch.Tensor) -> int:
    if t.dtype == torch.bfloat16:
        return DT_BF16
    if t.dtype == torch.float32:
        return DT_FP32
    if t.dtype == torch.float16:
        return DT_FP16
    raise DitangoHipError(f"unsupported state dtype {t.dtype} (bf16, fp16 or fp32)")


HALF_DTYPES = (torch.bfloat16, torch.float16)   # the 16-bit types the attention kernel runs in


def _require(cond: bool, msg: str) -> None:
    if not cond:
        raise DitangoHipError(msg)


def _check_qkv(q: torch.Tensor, name: str = "q", dtype: Optional[torch.dtype] = None) -> None:
    _require(q.is_cuda, f"{name} must live on the GPU")
    if dtype is None:
        _require(q.dtype in HALF_DTYPES, f"{name} must be bf16 or fp16 (got {q.dtype})")
    else:
        _require(q.dtype == dtype, f"{name} must be {dtype} like the other attention inputs (got {q.dtype})")
    _require(q.dim() == 4 and q.stride(-1) == 1, f"{name} must be [B,S,H,D] with contiguous D")


def _attn_flags(q: torch.Tensor, q_prescaled: bool) -> int:
    _require(q.dtype in HALF_DTYPES, f"the MFMA kernels take bf16 or fp16 tensors (got {q.dtype})")
    _require(not (q_prescaled and q.dtype == torch.float16), "a prescaled q is a bf16 mode")
    return (DT_ATTN_Q_PRESCALED if q_prescaled else 0) | (DT_ATTN_FP16 if q.dtype == torch.float16 else 0)


def lse_layout_of(lse: torch.Tensor, B: int, S: int, H: int) -> int:
    """Classify an lse tensor as [B,H,S] or [B,S,H(,1)] storage; it must be dense in that order.  Where the
    shape alone cannot tell (S == H), a 4-D tensor is read as the running layout [B,S,H,1] of utils.py:49 and a
    3-D tensor as flash-attn's [B,H,S]."""
    return _host().lse_layout(lse, B, S, H)


# ---------------------------------------------------------------------------------------------
# K1: chunk attention
# ---------------------------------------------------------------------------------------------

def attn_chunk_fwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, softmax_scale: float = 0.0,
                   out: Optional[torch.Tensor] = None, lse: Optional[torch.Tensor] = None):
    """(out [B,Sq,H,D] in q's dtype -- bf16 or fp16 --, lse fp32 [B,H,Sq]) of q against one KV chunk."""
    lib = load_library()
    _check_qkv(q, "q"); _check_qkv(k, "k", q.dtype); _check_qkv(v, "v", q.dtype)
    B, Sq, H, D = q.shape
    Sk = k.shape[1]
    _require(k.shape == v.shape and k.shape[0] == B and k.shape[2] == H and k.shape[3] == D, "k/v shape mismatch")
    _require(k.stride() == v.stride(), "k and v must share strides")
    if out is None:
        out = torch.empty((B, Sq, H, D), dtype=q.dtype, device=q.device)
    if lse is None:
        lse = torch.empty((B, H, Sq), dtype=torch.float32, device=q.device)
    _require(out.is_contiguous() and lse.is_contiguous() and out.dtype == q.dtype, "out/lse must be contiguous, out in q's dtype")
    fn = lib.dt_attn_chunk_f16_fwd if q.dtype == torch.float16 else lib.dt_attn_chunk_fwd
    rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(),
            B, Sq, Sk, H, D, q.stride(0), q.stride(1), q.stride(2),
            k.stride(0), k.stride(1), k.stride(2), float(softmax_scale), _stream())
    _check(rc, "dt_attn_chunk_fwd")
    return out, lse


def attn_chunk_f32_fwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, softmax_scale: float = 0.0):
    """(out fp32 [B,Sq,H,D], lse fp32 [B,H,Sq]) of fp32 q against one fp32 KV chunk, computed in fp32."""
    return attn_jobs_f32_fwd(q, [k], [v], [[0]], softmax_scale)[0]


def attn_jobs_f32_fwd(q: torch.Tensor, k_chunks: Sequence[torch.Tensor], v_chunks: Sequence[torch.Tensor],
                      jobs: Sequence[Sequence[int]], softmax_scale: float = 0.0, lse_bsh: bool = False) -> List[Tuple[torch.Tensor, torch.Tensor]]:
    """One launch: the fp32 states (out [B,Sq,H,D], lse [B,H,Sq] or, with ``lse_bsh``, [B,Sq,H,1]) of fp32 q against the
    concatenations of the fp32 chunks ``jobs[j]``.  Each chunk may have strides of its own.  More jobs or chunks than one
    launch addresses run in several.  Under graph capture workspace and counters come from the graph's pool, and every replay clears the
    counters."""
    _require(q.is_cuda and q.dim() == 4, "q must be fp32 [B,S,H,D] on the GPU with contiguous D")
    B, Sq, H, _ = q.shape
    need = len(jobs) * B * H * (-(-Sq // 32))
    counters = torch.zeros(need, dtype=torch.int32, device=q.device) if torch.cuda.is_current_stream_capturing() \
        else _stream_counters(q.device, need)
    return _host().attn_states_f32(q, k_chunks, v_chunks, jobs, softmax_scale, _stream(), lse_bsh, attn_workspace(q.device), counters)


_workspaces: "dict" = {}   # (device type, index, stream handle) -> tensor, in order of last use
MAX_WORKSPACES = 4         # streams per process that keep a workspace (about 102 MB each)


def attn_workspace(device) -> torch.Tensor:
    """The workspace of the attention launches made on the current stream of ``device`` (``dt_attn_workspace_bytes()``
    bytes).  Launches that share a workspace must be ordered on one stream; keyed by the stream, launches made on
    different streams never share one.  At most ``MAX_WORKSPACES`` streams keep theirs: the least recently used
    entry is dropped (its memory goes back to the allocator in stream order, so launches still in flight on that
    stream are safe).  A stream that is being captured in a graph uses none of them: a replay would write into a workspace that
    eager launches of that stream may be using at the same time, or that has been dropped since.  Launches under capture get
    memory of the graph's own pool, which the launches behind them reuse; the allocation-free entry point
    (``attn_jobs_fwd(..., no_alloc=True)``) needs none."""
    dev = device if isinstance(device, torch.device) else torch.device(device)
    if torch.cuda.is_current_stream_capturing():
        return torch.empty(int(load_library().dt_attn_workspace_bytes()), dtype=torch.uint8, device=dev)
    index = dev.index if dev.index is not None else torch.cuda.current_device()
    key = (dev.type, index, _raw_stream(index))
    ws = _workspaces.pop(key, None)
    if ws is None:
        while len(_workspaces) >= MAX_WORKSPACES:
            _workspaces.pop(next(iter(_workspaces)))
        ws = torch.empty(int(load_library().dt_attn_workspace_bytes()), dtype=torch.uint8, device=dev)
    _workspaces[key] = ws       # most recently used last
    return ws


_counters: "dict" = {}     # as _workspaces
KEPT_COUNTERS = 1 << 18    # words a kept set holds: launches of up to 32 512 query tiles


def attn_counters(device, q: torch.Tensor) -> Optional[torch.Tensor]:
    """The arrival counters of merging launches on ``q [B,Sq,H,D]`` made on the current stream of ``device``: int32, zero, and
    left at zero by every launch.  One set per stream, kept and shared like the workspace.  ``None``, and the launch does not
    merge, where it needs more than a kept set holds, and under capture: a graph's set would have to be cleared by every replay, a
    launch more than the merge saves."""
    B, Sq, H, _ = q.shape
    dev = device if isinstance(device, torch.device) else torch.device(device)
    return _stream_counters(dev, int(load_library().dt_attn_merge_counters(B, Sq, H)))


def _stream_counters(dev: torch.device, need: int) -> Optional[torch.Tensor]:
    """``attn_counters`` for a launch that needs ``need`` of them: what the native side calls when it is about to merge."""
    if need > KEPT_COUNTERS or torch.cuda.is_current_stream_capturing():
        return None
    index = dev.index if dev.index is not None else torch.cuda.current_device()
    key = (dev.type, index, _raw_stream(index))
    c = _counters.pop(key, None)
    if c is None:
        while len(_counters) >= MAX_WORKSPACES:
            _counters.pop(next(iter(_counters)))
        c = torch.empty(KEPT_COUNTERS, dtype=torch.int32, device=dev).zero_()
    _counters[key] = c
    return c


def attn_scratch(dev: torch.device):
    """``attn_workspace``, and the counters that the current stream keeps (``None``: it has none yet, or is being captured) for a caller
    that may merge: one look at the stream for both."""
    if torch.cuda.is_current_stream_capturing():
        return attn_workspace(dev), None
    index = dev.index if dev.index is not None else torch.cuda.current_device()
    key = (dev.type, index, _raw_stream(index))
    ws = _workspaces.pop(key, None)
    if ws is None:
        return attn_workspace(dev), None
    _workspaces[key] = ws
    c = _counters.pop(key, None)
    if c is not None:
        _counters[key] = c
    return ws, c


def release_workspaces() -> None:
    """Drop every attention workspace (they are re-created on demand)."""
    _workspaces.clear()
    _counters.clear()


class ChunkTable:
    """Host-side table of the KV chunks one layer call can touch (pointers, lengths, strides).  A table
    may hold more chunks than one launch can address (``DT_MAX_CHUNKS``); the job launches then pass the
    sub-table of the chunks their jobs reference.  ``batch``: 3-D chunks are packed ``[batch * S, H, D]``;
    ``convert`` is called on chunks that are neither bf16 nor fp16."""

    def __init__(self, k_chunks: Sequence[torch.Tensor], v_chunks: Sequence[torch.Tensor], batch: int = 0, convert=None):
        # (the binding takes sequences; a tensor of chunks or an iterator becomes one)
        k_chunks, v_chunks = (c if type(c) is list or type(c) is tuple else list(c) for c in (k_chunks, v_chunks))
        self.native = _host().ChunkTable(k_chunks, v_chunks, batch, convert)

    n = property(lambda self: self.native.n)
    B = property(lambda self: self.native.B)
    H = property(lambda self: self.native.H)
    D = property(lambda self: self.native.D)
    ss = property(lambda self: self.native.ss)
    sh = property(lambda self: self.native.sh)

    def whole(self):
        """ctypes arrays (k_ptrs, v_ptrs, lens, batch strides) of the whole table, for callers of the C ABI."""
        _require(self.n <= DT_MAX_CHUNKS, f"the table holds {self.n} chunks, one launch addresses {DT_MAX_CHUNKS}")
        return tuple((ct * self.n)(*xs) for ct, xs in zip((c_vp, c_vp, c_i32, c_i64), self.native.arrays))

    k_ptrs = property(lambda self: self.whole()[0])
    v_ptrs = property(lambda self: self.whole()[1])
    lens = property(lambda self: self.whole()[2])
    sb = property(lambda self: self.whole()[3])


def native_table(k_chunks: list, v_chunks: list, batch: int = 0, convert=None):
    """What ``ChunkTable(...).native`` is, for a caller that has lists and needs no more of the table."""
    return _host().ChunkTable(k_chunks, v_chunks, batch, convert)


class DeviceSegments:
    """Segment boundaries of a packed variable-length batch that live in device memory, as
    ``flash_attn_varlen_func`` takes them: ``cu_q`` int32 ``[n_seg + 1]`` for the queries and one such tensor
    per KV chunk for its keys (``cu_kv[c]``; ``None`` for a chunk without keys).  ``max_seqlen_q`` is the
    host-side upper bound of a segment's length that sizes the grid.  Nothing here reads device memory."""

    def __init__(self, cu_q: torch.Tensor, cu_kv: Sequence[Optional[torch.Tensor]], max_seqlen_q: int):
        self.cu_q = cu_q
        self.cu_kv = list(cu_kv)
        self.max_seqlen_q = int(max_seqlen_q)
        self.native = _host().Segments(cu_q, self.cu_kv, self.max_seqlen_q)
        self.n_seg = self.native.n_seg

    def window(self, w0: int, w1: int) -> "DeviceSegments":
        return DeviceSegments(self.cu_q, self.cu_kv[w0:w1], self.max_seqlen_q)


def attn_jobs_fwd(q: torch.Tensor, table: ChunkTable, jobs: Sequence[Sequence[int]],
                  outs: Sequence[torch.Tensor], lses: Sequence[torch.Tensor], softmax_scale: float = 0.0,
                  q_ranges: Optional[Sequence[Tuple[int, int]]] = None,
                  kv_ranges: Optional[Sequence[Sequence[Tuple[int, int]]]] = None,
                  workspace: Optional[torch.Tensor] = None, q_prescaled: bool = False,
                  no_alloc: bool = False, dev_segments: Optional["DeviceSegments"] = None,
                  job_segments: Optional[Sequence[int]] = None) -> None:
    """One launch; job j attends q to the concatenation of chunks ``jobs[j]`` and writes (outs[j], lses[j]).

    ``q_ranges[j] = (begin, length)`` restricts job j to those query rows (the rest of its
    destination is left untouched); ``kv_ranges[j][i] = (begin, length)`` restricts the i-th chunk
    of job j to those keys.  Several jobs may share one destination if their rows are disjoint
    (the segments of a packed variable-length batch).  Launches are split to respect the limits
    of one launch.  With a ``workspace`` (``attn_workspace(device)``) the last, partly filled round of
    workgroups of a launch is split along the keys and folded back (tail balancing).
    ``q_prescaled``: q already carries ``softmax_scale * log2(e)`` (folded in before its rounding to
    bf16); ``softmax_scale`` is then ignored and the softmax is that of ``q k^T * ln 2``.
    ``no_alloc``: go through ``dt_attn_seg_jobs_noalloc_fwd``, which splits the tail inside the library's
    own device array instead of a workspace (for callers that cannot allocate).
    ``dev_segments`` with ``job_segments``: the segment boundaries stay in device memory
    (``dt_attn_varlen_jobs_fwd``); job j is segment ``job_segments[j]`` of its state and the host reads none
    of the boundaries."""
    _host().attn_jobs(q, table.native, jobs, outs, lses, softmax_scale, q_ranges, kv_ranges, workspace,
                      _attn_flags(q, q_prescaled), no_alloc, None if dev_segments is None else dev_segments.native,
                      job_segments, _stream())


def attn_states(q: torch.Tensor, k_chunks: Sequence[torch.Tensor], v_chunks: Sequence[torch.Tensor],
                jobs: Sequence[Sequence[int]], max_chunks: int, workspace: Optional[torch.Tensor] = None,
                q_prescaled: bool = False, cu_q: Optional[Sequence[int]] = None,
                cu_kv: Optional[Sequence[Sequence[int]]] = None, dev_segments: Optional[DeviceSegments] = None,
                convert=None) -> List[Tuple[torch.Tensor, torch.Tensor]]:
    """The fresh states (out [B,Sq,H,D] in q's dtype, lse [B,H,Sq]) of q against the concatenations of the chunks
    ``jobs[j]``, computed in one launch where its limits allow.  A job of more than ``max_chunks`` chunks is computed in
    pieces.  A packed variable-length batch brings its boundaries as host lists (``cu_q``, ``cu_kv[chunk]``) or as
    ``dev_segments``; rows outside every segment are left as they are.  ``convert`` as in ``ChunkTable``."""
    return _host().attn_states(q, k_chunks, v_chunks, jobs, max_chunks, cu_q, cu_kv, workspace, _attn_flags(q, q_prescaled),
                               None if dev_segments is None else dev_segments.native, convert, _stream())


def attn_states_merge(q: torch.Tensor, k_chunks: Sequence[torch.Tensor], v_chunks: Sequence[torch.Tensor],
                      jobs: Sequence[Sequence[int]], max_chunks: int, outs: Sequence[torch.Tensor], lses: Sequence[torch.Tensor],
                      which: Sequence[int], dst_dtype: torch.dtype, workspace: Optional[torch.Tensor] = None,
                      q_prescaled: bool = False, cu_q: Optional[Sequence[int]] = None,
                      cu_kv: Optional[Sequence[Sequence[int]]] = None, dev_segments: Optional[DeviceSegments] = None,
                      convert=None):
    """``attn_states``, and the merge of the given states and then ``states[which[..]]`` (``merge_states`` with a
    ``[B,S,H,1]`` lse), in the same launch where it can.  Returns (states, out, lse)."""
    return _host().attn_states_merge(q, k_chunks, v_chunks, jobs, max_chunks, cu_q, cu_kv, workspace, _attn_flags(q, q_prescaled),
                                     None if dev_segments is None else dev_segments.native, convert, outs, lses, which, dst_dtype,
                                     lambda need: _stream_counters(q.device, need), _stream())


def attn_sched_merge(q: torch.Tensor, table, dev_compute_ids: torch.Tensor, dev_count: torch.Tensor, max_jobs: int,
                     slot_out: torch.Tensor, slot_lse: torch.Tensor, diag: int, diag_out: torch.Tensor, diag_lse: torch.Tensor,
                     dst_dtype: torch.dtype, workspace: Optional[torch.Tensor] = None, q_prescaled: bool = False, row: int = 0,
                     counters: Optional[torch.Tensor] = None):
    """``attn_sched_fwd`` on whole queries and ``merge_arena``, in the same launch where it can.  ``table`` is a ``ChunkTable`` or a
    ``native_table``; ``counters`` those that ``attn_scratch`` found for this stream.  Returns (out, lse)."""
    return _host().attn_sched_merge(q, table.native if type(table) is ChunkTable else table, dev_compute_ids, dev_count, row, max_jobs, slot_out, slot_lse, diag, diag_out,
                                    diag_lse, dst_dtype, workspace,
                                    (lambda need: _stream_counters(q.device, need)) if counters is None else counters,
                                    _attn_flags(q, q_prescaled), _stream())


def attn_sched_fwd(q: torch.Tensor, table: ChunkTable, dev_compute_ids: torch.Tensor, dev_count: torch.Tensor,
                   max_jobs: int, slot_out: torch.Tensor, slot_lse: torch.Tensor, diag: int,
                   diag_out: Optional[torch.Tensor], diag_lse: Optional[torch.Tensor],
                   softmax_scale: float = 0.0, seg_q: Optional[Sequence[Tuple[int, int]]] = None,
                   seg_kv: Optional[Sequence[Sequence[Tuple[int, int]]]] = None,
                   workspace: Optional[torch.Tensor] = None, q_prescaled: bool = False,
                   dev_segments: Optional[DeviceSegments] = None, row: int = 0) -> None:
    """Device-scheduled launch: chunk ids come from ``dev_compute_ids[:dev_count]`` in device memory (of a whole
    schedule, ``[..., C]`` and ``[..., 2]``: from its row ``row``) and
    each state lands in its slot of the arena (``slot_out [C,B,Sq,H,D]`` in q's dtype, ``slot_lse [C,B,H,Sq]`` fp32).

    On a packed variable-length batch, ``seg_q[s] = (begin, length)`` are the query rows of segment s and
    ``seg_kv[c][s] = (begin, length)`` its keys inside chunk c; every scheduled chunk then runs once per segment."""
    _host().attn_sched(q, table.native, dev_compute_ids, dev_count, row, max_jobs, slot_out, slot_lse, diag, diag_out, diag_lse,
                       softmax_scale, seg_q, seg_kv, workspace, _attn_flags(q, q_prescaled),
                       None if dev_segments is None else dev_segments.native, _stream())


# ---------------------------------------------------------------------------------------------
# K2: merge, K3: cache store/load
# ---------------------------------------------------------------------------------------------

def merge_states(outs: Sequence[torch.Tensor], lses: Sequence[torch.Tensor],
                 dst_out: Optional[torch.Tensor] = None, dst_lse: Optional[torch.Tensor] = None,
                 dst_dtype: torch.dtype = torch.float32, dst_lse_bsh: bool = False):
    """N-way LSE merge.  outs[i] contiguous [B,Sq,H,D] (bf16, fp16 or fp32, in any mix), lses[i] fp32 in
    [B,H,Sq] or [B,Sq,H(,1)] storage.  Returns (dst_out, dst_lse).  Up to ``DT_MAX_MERGE`` states are one
    pass over HBM; more are folded in rounds through a running fp32 state that is updated in place (the
    merge is associative; the running state is never rounded below fp32)."""
    return _host().merge(outs, lses, dst_out, dst_lse, dst_dtype, dst_lse_bsh, _stream())


def merge_arena(arena_out: torch.Tensor, arena_lse: torch.Tensor, diag: int, diag_out: torch.Tensor, diag_lse: torch.Tensor,
                dst_dtype: torch.dtype = torch.float32):
    """Merge of every slot of an arena ``[C,B,Sq,H,D]`` / ``[C,B,H,Sq]``, slot ``diag`` replaced by
    (diag_out, diag_lse).  Returns (out ``[B,Sq,H,D]``, lse ``[B,Sq,H,1]``)."""
    return _host().merge_arena(arena_out, arena_lse, diag, diag_out, diag_lse, dst_dtype, _stream())


def cache_store(src_out: torch.Tensor, src_lse: torch.Tensor, slot_out: torch.Tensor, slot_lse: torch.Tensor) -> None:
    _host().cache_store(src_out, src_lse, slot_out, slot_lse, _stream())


def cache_load(slot_out: torch.Tensor, slot_lse: torch.Tensor, dst_dtype: torch.dtype = torch.float32,
               dst_lse_bsh: bool = False, dst_out: Optional[torch.Tensor] = None, dst_lse: Optional[torch.Tensor] = None):
    return _host().cache_load(slot_out, slot_lse, dst_dtype, dst_lse_bsh, dst_out, dst_lse, _stream())


def zero_rows_from(t: torch.Tensor, first_row: torch.Tensor) -> None:
    """Zero the rows ``[first_row[0], n)`` of ``t`` (contiguous, rows along dim 0), the index read on the device."""
    _host().zero_rows_from(t, first_row, _stream())


# ---------------------------------------------------------------------------------------------
# K4: schedule builder, rel-L1 sums
# ---------------------------------------------------------------------------------------------

def build_schedule(mask: torch.Tensor, t: int, l: int, diag: int = -1):
    """(compute_ids [C], reuse_ids [C], counts [2]) int32 device tensors for row (t, l) of mask uint8 [T,L,C]."""
    lib = load_library()
    _require(mask.is_cuda and mask.dtype == torch.uint8 and mask.dim() == 3 and mask.is_contiguous(), "mask must be contiguous uint8 [T,L,C] on the GPU")
    T, L, C = mask.shape
    comp = torch.empty(C, dtype=torch.int32, device=mask.device)
    reu = torch.empty(C, dtype=torch.int32, device=mask.device)
    cnt = torch.empty(2, dtype=torch.int32, device=mask.device)
    rc = lib.dt_build_schedule(mask.data_ptr(), T, L, C, int(t), int(l), int(diag), comp.data_ptr(), reu.data_ptr(), cnt.data_ptr(), _stream())
    _check(rc, "dt_build_schedule")
    return comp, reu, cnt


def build_schedule_table(mask: torch.Tensor, diag: int = -1):
    lib = load_library()
    _require(mask.is_cuda and mask.dtype == torch.uint8 and mask.dim() == 3 and mask.is_contiguous(), "mask must be contiguous uint8 [T,L,C] on the GPU")
    T, L, C = mask.shape
    comp = torch.empty((T, L, C), dtype=torch.int32, device=mask.device)
    reu = torch.empty((T, L, C), dtype=torch.int32, device=mask.device)
    cnt = torch.empty((T, L, 2), dtype=torch.int32, device=mask.device)
    rc = lib.dt_build_schedule_table(mask.data_ptr(), T, L, C, int(diag), comp.data_ptr(), reu.data_ptr(), cnt.data_ptr(), _stream())
    _check(rc, "dt_build_schedule_table")
    return comp, reu, cnt


def rel_l1_sums(a: torch.Tensor, b: torch.Tensor, sums: Optional[torch.Tensor] = None) -> torch.Tensor:
    """fp64 [4] device tensor: sum|a-b|, sum|a|, sum|b|, count over entries where neither is NaN (no host sync)."""
    lib = load_library()
    _require(a.is_cuda and b.is_cuda and a.dtype == torch.float32 and b.dtype == torch.float32, "inputs must be fp32 on the GPU")
    _require(a.is_contiguous() and b.is_contiguous() and a.numel() == b.numel(), "inputs must be contiguous and equally sized")
    if sums is None:
        sums = torch.zeros(4, dtype=torch.float64, device=a.device)
    rc = lib.dt_rel_l1_sums(a.data_ptr(), b.data_ptr(), a.numel(), sums.data_ptr(), _stream())
    _check(rc, "dt_rel_l1_sums")
    return sums


def qk_norm_rope(x: torch.Tensor, *, norm: int = DT_NORM_NONE, weight: Optional[torch.Tensor] = None,
                 bias: Optional[torch.Tensor] = None, eps: float = 1e-6, rope: int = DT_ROPE_NONE,
                 cos: Optional[torch.Tensor] = None, sin: Optional[torch.Tensor] = None,
                 rope_begin: int = 0, rope_end: Optional[int] = None, sections: Sequence[int] = (),
                 rounding: int = 0, out: Optional[torch.Tensor] = None, out_scale: float = 1.0) -> torch.Tensor:
    """x bf16 or fp16 ``[B,S,H,D]`` (any strides with a contiguous last dimension) -> ``[B,S,H,D]`` contiguous in
    the same dtype, normalised over D and rotated on token rows ``[rope_begin, rope_end)``.  cos/sin are fp32
    ``[rope_end-rope_begin, D]`` or ``[B, rope_end-rope_begin, D]``.  ``out_scale`` multiplies the result
    before its rounding to the output dtype; the ``DT_ROUND_*`` bits round to x's dtype.  weight / bias are fp32, or
    with ``DT_WEIGHTS_16`` in ``rounding`` of x's dtype."""
    _require(x.is_cuda, "x must be bf16 or fp16 [B,S,H,D] on the GPU")   # (before a stream is asked for)
    # (the binding takes no float for a whole number and no array for a list)
    return _host().qk_norm_rope(x, int(norm), weight, bias, float(eps), int(rope), cos, sin, int(rope_begin),
                                None if rope_end is None else int(rope_end), [int(v) for v in sections], int(rounding), out, float(out_scale),
                                _stream())


def qkv_project(text: torch.Tensor, video: torch.Tensor, heads: int, projections, cos: Optional[torch.Tensor] = None,
                sin: Optional[torch.Tensor] = None):
    """q, k and v ``[B,T+V,heads,64]`` of ``text`` ``[B,T,K]`` and ``video`` ``[B,V,K]`` in one launch.  ``projections``: three of
    ``(weight, bias, norm, norm_weight, norm_bias, eps, rope)``; cos/sin fp32 ``[V,64]`` for those with ``rope``."""
    return _host().qkv_project(text, video, heads, projections, cos, sin, _stream())
