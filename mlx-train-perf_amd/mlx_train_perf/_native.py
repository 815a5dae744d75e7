"""ctypes binding of the HIP C-ABI library (``libmtp_hip.so``, declared in ``include/mtp_hip.h``).

This is the only place the package touches native code. The library is built in-tree by
``__graft_entry__.build()`` (or ``python -m mlx_train_perf._build``) for gfx950. There is no fallback:
if the library is missing or no GPU is visible, the kernel impls raise ``MissingDependencyError`` /
``UnsupportedHeadError`` / ``UnsupportedAttentionError`` before any launch.

torch must be imported before the library is loaded so that the process holds exactly one HIP
runtime (torch's): the library's ``libamdhip64.so.7`` dependency then resolves to the copy torch
already mapped, and torch's stream handles are valid for our launches.
"""
from __future__ import annotations

import ctypes
import os
import threading
import warnings
from pathlib import Path

import torch
from torch.autograd import forward_ad

from mlx_train_perf.errors import (
    AttentionInputError,
    LaunchBudgetError,
    LossInputError,
    MissingDependencyError,
    MlxTrainPerfError,
    UnsupportedAttentionError,
    UnsupportedHeadError,
)

LIB_NAME = "libmtp_hip.so"
LIB_PATH = Path(os.environ.get("MTP_HIP_LIB", str(Path(__file__).resolve().parent / LIB_NAME)))

ABI_VERSION = 5
MTP_OK = 0
MTP_ERR_INPUT = -1
MTP_ERR_UNSUPPORTED = -2
MTP_ERR_WORKSPACE = -3
MTP_ERR_RUNTIME = -4

HEAD_DENSE = 0
HEAD_Q4 = 1
HEAD_Q4_STAGED = 2      # kinds that stage the head chunk-wise in the workspace: the backward each
HEAD_DENSE_STAGED = 3   # transposed (4-bit: dequantized) vocab chunk instead of a cached transposed
                        # copy, the 4-bit forward runs of vocab splits dequantized to rows

_c_void_p = ctypes.c_void_p
_i64 = ctypes.c_int64
_i32 = ctypes.c_int32
_f32 = ctypes.c_float
_size = ctypes.c_size_t

# name -> (restype, argtypes); the single source of truth for the Python side of the ABI.
SIGNATURES: dict[str, tuple[object, list[object]]] = {
    "mtp_last_error": (ctypes.c_char_p, []),
    "mtp_abi_version": (ctypes.c_int, []),
    "mtp_lce_fwd_workspace_bytes": (_size, [_i64, _i64, _i64, _i32]),
    "mtp_lce_fwd_stage_workspace_bytes": (_size, [_i64, _i64, _i64, _size]),
    "mtp_lce_fwd": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,
                                   _i64, _i64, _i64, _i32, _i64, _c_void_p, _c_void_p, _c_void_p,
                                   _c_void_p, _size, _c_void_p]),
    "mtp_lce_fwd_noalloc": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,
                                           _i64, _i64, _i64, _i32, _i64, _c_void_p, _c_void_p, _c_void_p,
                                           _c_void_p]),
    "mtp_lce_fwd_noalloc_max_workspace_bytes": (_size, []),
    "mtp_lce_bwd_row_block": (_i64, [_i64, _i64, _i64, _size]),
    "mtp_lce_bwd_chunk": (_i64, [_i64, _i64, _i64, _size]),
    "mtp_lce_bwd_stage_chunk": (_i64, [_i64, _i64, _i64, _i32, _size]),
    "mtp_lce_bwd_workspace_bytes": (_size, [_i64, _i64, _i64, _i32, _i64, _i64]),
    "mtp_lce_head_t_ld": (_i64, [_i64]),
    "mtp_lce_head_transpose": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _i64, _i64, _i32,
                                              _c_void_p, _c_void_p]),
    "mtp_lce_bwd": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,
                                   _i64, _i64, _i64, _i32, _i64, _c_void_p, _c_void_p, _c_void_p,
                                   _c_void_p, _i64, _i64, _c_void_p, _size, _c_void_p]),
    "mtp_lce_mean": (ctypes.c_int, [_c_void_p, _c_void_p, _i64, _i64, _c_void_p, _c_void_p, _c_void_p]),
    "mtp_lce_mean_bwd": (ctypes.c_int, [_c_void_p, _c_void_p, _i64, _c_void_p, _c_void_p]),
    "mtp_attn_fwd": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _i64, _i64, _i64, _i64, _i64,
                                    _f32, _i32, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p]),
    "mtp_attn_bwd_workspace_bytes": (_size, [_i64, _i64, _i64, _i64, _i64]),
    "mtp_attn_bwd_dkv_splits": (ctypes.c_int, [_i64, _i64, _i64, _i64, _i64, _i32]),
    "mtp_bench_mfma_ceiling": (ctypes.c_int, [ctypes.c_int, ctypes.c_int, _c_void_p, _c_void_p]),
    "mtp_attn_bwd": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,
                                    _i64, _i64, _i64, _i64, _i64, _f32, _i32, _c_void_p, _c_void_p,
                                    _c_void_p, _c_void_p, _c_void_p, _c_void_p, _size, _c_void_p]),
    # fp32 inputs
    "mtp_lce_fwd_f32_workspace_bytes": (_size, [_i64, _i64, _i64, _i32]),
    "mtp_lce_fwd_f32": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,
                                       _i64, _i64, _i64, _i32, _i64, _c_void_p, _c_void_p, _c_void_p,
                                       _c_void_p, _size, _c_void_p]),
    "mtp_lce_bwd_f32_chunk": (_i64, [_i64, _i64, _i64, _size]),
    "mtp_lce_bwd_f32_workspace_bytes": (_size, [_i64, _i64, _i64, _i64]),
    "mtp_lce_bwd_f32": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,
                                       _i64, _i64, _i64, _i32, _i64, _c_void_p, _c_void_p, _c_void_p,
                                       _c_void_p, _i64, _c_void_p, _size, _c_void_p]),
    "mtp_attn_fwd_f32": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _i64, _i64, _i64, _i64, _i64,
                                        _f32, _i32, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p]),
    "mtp_attn_bwd_f32_workspace_bytes": (_size, [_i64, _i64, _i64, _i64, _i64]),
    "mtp_attn_bwd_f32": (ctypes.c_int, [_c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,
                                        _i64, _i64, _i64, _i64, _i64, _f32, _i32, _c_void_p, _c_void_p,
                                        _c_void_p, _c_void_p, _c_void_p, _c_void_p, _size, _c_void_p]),
}

_lock = threading.Lock()
_lib: ctypes.CDLL | None = None


def load() -> ctypes.CDLL:
    """Load (once) and return the library with typed signatures; raise if it is absent."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not LIB_PATH.exists():
            raise MissingDependencyError(
                f"HIP extension {LIB_PATH} is not built; run `python -c \"import __graft_entry__ as g; "
                "g.build()\"` from the repository root (hipcc --offload-arch=gfx950)."
            )
        lib = ctypes.CDLL(str(LIB_PATH), mode=ctypes.RTLD_GLOBAL)
        version = lib.mtp_abi_version() if hasattr(lib, "mtp_abi_version") else None
        if version != ABI_VERSION:
            raise MissingDependencyError(f"{LIB_PATH} has ABI version {version}, expected {ABI_VERSION}; rebuild it")
        missing = [name for name in SIGNATURES if not hasattr(lib, name)]
        if missing:   # an older build of this version, which grows by new exports
            raise MissingDependencyError(f"{LIB_PATH} does not export {', '.join(missing)}; rebuild it")
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _lib = lib
        return lib


_nodes = None   # the module once loaded, False where it cannot be


def nodes():
    """Load (once) and return the extension module with the autograd nodes (csrc/torch_nodes.cpp), bound to
    the loaded library's entry points. None where it was not built, or (with a warning) where it does not
    load, as when it was built against another torch: the Python Functions then serve every call, the same
    bits for more host time."""
    global _nodes
    if _nodes is None:
        lib = load()
        with _lock:
            if _nodes is None:
                _nodes = _bind_nodes(lib)
    return _nodes or None


def _bind_nodes(lib):
    try:
        from mlx_train_perf import _mtp_torch
    except ImportError as e:
        path = Path(__file__).with_name("_mtp_torch.so")
        if path.exists():
            warnings.warn(f"{path} cannot be loaded ({e}); calls take the Python autograd functions. Run "
                          "`python -c \"import __graft_entry__ as g; g.build()\"` from the repository root.", stacklevel=2)
        return False
    from mlx_train_perf.attention import api
    from mlx_train_perf.core import loss
    from mlx_train_perf.plan import launch

    _mtp_torch.bind({name: ctypes.cast(getattr(lib, name), _c_void_p).value for name in SIGNATURES}, check)
    _mtp_torch.bind_attention(api.VJP_CALLS)
    _mtp_torch.bind_loss(loss.VJP_CALLS, loss._transposed_head, launch.lce_bwd_budget_bytes, os.environ.get)
    return _mtp_torch


def plain(*tensors: torch.Tensor) -> bool:
    """Ordinary tensors outside function transforms, tracing and dispatch modes, without a forward-mode
    tangent: the calls that the C++ nodes take. The others keep the Python Functions, which refuse or
    serve them as they always did (a node sees no tangent of a tensor that is not its input)."""
    return (all(type(t) in (torch.Tensor, torch.nn.Parameter) for t in tensors)
            and not torch._C._are_functorch_transforms_active() and torch._C._get_tracing_state() is None
            and not torch.compiler.is_compiling() and torch._C._len_torch_dispatch_stack() == 0
            and (forward_ad._current_level < 0 or all(forward_ad.unpack_dual(t).tangent is None for t in tensors)))


def gpu_available() -> bool:
    return torch.cuda.is_available()


def last_error() -> str:
    msg = load().mtp_last_error()
    return msg.decode() if msg else ""


_ERR_LOSS = {MTP_ERR_INPUT: LossInputError, MTP_ERR_UNSUPPORTED: UnsupportedHeadError,
             MTP_ERR_WORKSPACE: LaunchBudgetError}
_ERR_ATTN = {MTP_ERR_INPUT: AttentionInputError, MTP_ERR_UNSUPPORTED: UnsupportedAttentionError,
             MTP_ERR_WORKSPACE: LaunchBudgetError}


def check(rc: int, *, domain: str) -> None:
    """Map a negative C-ABI return code onto the reference's typed exceptions."""
    if rc == MTP_OK:
        return
    table = _ERR_LOSS if domain == "loss" else _ERR_ATTN
    exc = table.get(rc, MlxTrainPerfError)
    raise exc(last_error() or f"mtp call failed with code {rc}")


def ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def stream_of(t: torch.Tensor) -> int:
    # current_stream(t.device).cuda_stream without the Stream object it builds on every call
    return torch._C._cuda_getCurrentRawStream(t.device.index)


def on_device(t: torch.Tensor):
    """Context that makes t's GPU the current device for a C-ABI call. The launches go to t's stream;
    HIP calls inside the library that act on the current device (the no-allocation forward's scratch
    lookup, error queries) then see the same device whatever the caller had current."""
    return torch.cuda.device(t.device)
