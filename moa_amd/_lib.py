"""ctypes binding of libmoa_hip.so (declared in include/moa_hip.h).

There is no fallback: if the library is missing or does not load, every
operator of this package raises.  (The compiled host side, _host.so, which
makes the same calls of the library, may be missing: see host().)
"""
from __future__ import annotations

import ctypes
import os
import sys
import warnings
from ctypes import POINTER, c_char_p, c_float, c_int, c_int64, c_size_t, c_void_p
from typing import Optional, Sequence

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libmoa_hip.so")
HOST_PATH = os.path.join(HERE, "_host.so")

MOA_OK = 0
MOA_ERR_ARG = -1
MOA_ERR_UNSUPPORTED = -2
MOA_ERR_LAUNCH = -3
MOA_ERR_WORKSPACE = -4

MOA_DTYPE_F16 = 0
MOA_DTYPE_BF16 = 1
MOA_DTYPE_F32 = 2

MOA_DECODE_NOALLOC_MAX_BYTES = 32 << 20

ABI_VERSION = 1

# name -> (restype, argtypes); must list every symbol include/moa_hip.h declares
_I64P = POINTER(c_int64)
SIGNATURES = {
    "moa_abi_version": (c_int, []),
    "moa_last_error": (c_char_p, []),
    "moa_prefill_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, _I64P, _I64P, _I64P, _I64P,
                                c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_float, c_int,
                                c_void_p]),
    "moa_prefill_fwd_tokens": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, _I64P, _I64P, _I64P, _I64P,
                                       c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_float, c_int,
                                       c_void_p]),
    "moa_decode_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int64]),
    "moa_decode_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_size_t, c_void_p,
                               c_void_p, c_int, c_int, c_int, c_int, c_int64, c_float, c_int, c_void_p]),
    "moa_decode_fwd_counted": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_size_t, c_void_p,
                                       c_size_t, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int64, c_float,
                                       c_int, c_void_p]),
    "moa_decode_fwd_noalloc": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int,
                                       c_int, c_int, c_int64, c_float, c_int, c_void_p]),
    "moa_cache_append": (c_int, [c_void_p, c_void_p, _I64P, _I64P, c_void_p, c_void_p, c_void_p, c_void_p,
                                 c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int, c_int,
                                 c_int, c_int64, c_int, c_void_p]),
    "moa_cache_prefill_workspace_bytes": (c_size_t, [c_int, c_int]),
    "moa_cache_prefill_insert": (c_int, [c_void_p, c_void_p, _I64P, _I64P, c_void_p, c_void_p, c_void_p,
                                         c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64,
                                         c_void_p, c_size_t, c_int64, c_int, c_int, c_int, c_int, c_int64,
                                         c_int64, c_int, c_void_p]),
    "moa_rope_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, _I64P, _I64P, _I64P, _I64P, c_void_p,
                             c_void_p, _I64P, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p]),
    "moa_rope_cache_append": (c_int, [c_void_p, c_void_p, c_void_p, _I64P, _I64P, _I64P, c_void_p, c_void_p,
                                      c_int64, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                      c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int, c_int, c_int,
                                      c_int, c_int64, c_int, c_void_p]),
    "moa_rope_prefill_insert": (c_int, [c_void_p] * 5 + [_I64P] * 5 + [c_void_p, c_void_p, _I64P] + [c_void_p] * 9
                                + [c_int64, c_void_p, c_size_t, c_int64, c_int, c_int, c_int, c_int, c_int, c_int64,
                                   c_int64, c_int, c_int, c_void_p]),
}

_lib: Optional[ctypes.CDLL] = None
_host = None


class MoaKernelError(RuntimeError):
    """The HIP library is missing, or a launch failed."""


def load() -> ctypes.CDLL:
    """Loads the library once; raises MoaKernelError when it cannot."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise MoaKernelError(
            f"{LIB_PATH} is not built. Run `python -m moa_amd.build` (needs hipcc). "
            "moa_amd has no CPU or PyTorch fallback for its kernels.")
    try:
        lib = ctypes.CDLL(LIB_PATH)
    except OSError as e:  # pragma: no cover - depends on the machine
        raise MoaKernelError(f"cannot load {LIB_PATH}: {e}") from e
    for name, (res, args) in SIGNATURES.items():
        try:
            fn = getattr(lib, name)
        except AttributeError as e:
            raise MoaKernelError(f"{LIB_PATH} does not export {name}; rebuild it") from e
        fn.restype = res
        fn.argtypes = args
    v = lib.moa_abi_version()
    if v != ABI_VERSION:
        raise MoaKernelError(f"{LIB_PATH} has ABI version {v}, this package expects {ABI_VERSION}; rebuild it")
    _lib = lib
    return lib


def host_is_built_for() -> str:
    """What the compiled host side has to be built for to be loaded here: it uses torch's C++ classes and Python's."""
    import torch

    return f"torch {torch.__version__}, Python {sys.version_info[0]}.{sys.version_info[1]}"


def host_fits() -> bool:
    """Is there a compiled host side, and was it built for this torch and Python?  (Looked up in the file: one that was not is
    not loaded.)"""
    try:
        with open(HOST_PATH, "rb") as f:
            return f"moa_host was built for {host_is_built_for()};".encode() in f.read()
    except OSError:
        return False


class _NoHost:
    """Takes no call: the Python code behind it takes all of them, through ctypes."""
    attend = rope_append = append = staticmethod(lambda *args: None)


def host():
    """The compiled host side of the attention and the append (csrc/moa_host.cpp), loaded once and bound to the library.
    It only saves time.  Where it is missing or was built for another torch, the calls go through the Python code."""
    global _host
    if _host is not None:
        return _host
    import torch  # noqa: F401  (its libraries are what the module is linked to)

    lib = load()
    module, why = None, "is not built for " + host_is_built_for()
    if host_fits():
        try:
            from moa_amd import _host as module
        except ImportError as e:
            why = f"cannot be loaded ({e})"
    if module is None:
        warnings.warn(f"{HOST_PATH} {why}: small calls take the host longer. Run `python -m moa_amd.build`.", RuntimeWarning)
        _host = _NoHost
        return _host
    from moa_amd.kernels import mixture_of_attention as attention

    raw = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (lambda i: torch.cuda.current_stream(i).cuda_stream)
    module.setup(*(ctypes.cast(getattr(lib, f), c_void_p).value for f in (
        "moa_decode_workspace_bytes", "moa_decode_fwd_counted", "moa_rope_cache_append", "moa_cache_append",
        "moa_prefill_fwd_tokens")), raw, check, attention._decode_scratch, attention._N_COUNTERS)
    _host = module
    return module


def last_error() -> str:
    return load().moa_last_error().decode("utf-8", "replace")


def check(rc: int, assertion_for_arg: bool = True) -> None:
    """Maps a return code to the exception class the reference raises for the
    same condition: AssertionError for shape/dtype problems
    (MoA/kernels/mixture_of_attention.py:216,227,316), NotImplementedError for
    paths that are not covered (:478-479,486-487)."""
    if rc == MOA_OK:
        return
    msg = last_error()
    if rc == MOA_ERR_ARG and assertion_for_arg:
        raise AssertionError(msg)
    if rc == MOA_ERR_UNSUPPORTED:
        raise NotImplementedError(msg)
    raise MoaKernelError(f"libmoa_hip error {rc}: {msg}")


def i64_array(values: Sequence[int]):
    return (c_int64 * len(values))(*values)


def dtype_code(torch_dtype) -> int:
    import torch

    if torch_dtype == torch.float16:
        return MOA_DTYPE_F16
    if torch_dtype == torch.bfloat16:
        return MOA_DTYPE_BF16
    if torch_dtype == torch.float32:
        return MOA_DTYPE_F32
    raise AssertionError(f"unsupported dtype {torch_dtype}")


def current_stream_ptr(device) -> int:
    """The raw HIP stream torch is currently using on ``device`` (through torch's internal accessor
    when it exists: the public ``torch.cuda.current_stream`` costs several microseconds per call)."""
    import torch

    raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)
    if raw is not None:
        return raw(device.index if device.index is not None else torch.cuda.current_device())
    return torch.cuda.current_stream(device).cuda_stream


def ptr(t) -> Optional[int]:
    return None if t is None else t.data_ptr()
