"""ctypes binding of the C ABI in include/prime_decode.h (libprime_decode.so), and the host module
that checks and launches a decode step (csrc/host_step.cpp).

This is the only place Python crosses into native code.  There is no fallback for the library: if it
is missing its first use raises.  The host module is compiled against one torch and one Python; under
others decode_step makes the same checks in Python.
"""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import sysconfig
import warnings
from pathlib import Path

LIB_PATH = Path(__file__).resolve().parent / "_lib" / "libprime_decode.so"

MODEL_360M = 360
MODEL_135M = 135

# status codes of include/prime_decode.h that callers act on
PK_ERR_ABORTED = 9113
PK_ERR_NOALLOC = 9115
# pk_set_option options
PK_OPT_COOPERATIVE = 1
PK_OPT_SPLIT_ROLE = 2
PK_OPT_L2_RECORDS = 3
PK_OPT_SKEW = 4
PK_OPT_SPLIT_WIDE = 5

_lib = None
_host = None

vp, ci, ll, sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_longlong, ctypes.c_size_t

# symbol -> (restype, argtypes); the list every test checks against include/*.h
SIGNATURES = {
    "pk_workspace_bytes": (sz, [ci]),
    "pk_init": (ci, []),
    "pk_set_option": (ci, [ci, ci]),
    "pk_state_read": (ci, [vp, sz, ctypes.POINTER(ctypes.c_uint), ci]),
    "pk_state_status": (ci, [vp, ctypes.POINTER(ctypes.c_uint)]),
    "pk_state_take": (ci, [vp, ctypes.POINTER(ctypes.c_uint)]),
    "pk_test_exchange_units": (ci, [ci, ci, ci, ctypes.POINTER(ctypes.c_uint)]),
    "pk_test_set_epoch": (ci, [vp, ctypes.c_uint]),
    "pk_test_abort_next": (ci, [vp]),
    "pk_test_abort_next_noalloc": (ci, [vp]),
    "pk_noalloc_status": (ci, [vp, ci, ctypes.POINTER(ctypes.c_uint)]),
    "pk_decode": (ci, [vp, ci, ci, ci, vp, ci, vp, vp, vp, vp, vp, ci, vp, vp, vp,
                       ll, ll, ll, ll, ll, ci, vp, ci, vp, vp, vp, vp, vp, sz, ci]),
    "pk_decode_noalloc": (ci, [vp, ci, ci, ci, vp, ci, vp, vp, vp, vp, vp, ci, vp, vp, vp,
                               ll, ll, ll, ll, ll, ci, vp, ci, vp, vp, vp, vp, ci]),
    "pk_decode_debug": (ci, [vp, ci, ci, ci, vp, ci, vp, vp, vp, vp, vp, ci, vp, vp, vp,
                             ll, ll, ll, ll, ll, ci, vp, ci, vp, vp, vp, vp, vp, sz, ci, vp, vp, sz, ci]),
    "pk_decode_mxfp8": (ci, [vp, ci, ci, ci, vp, ci, vp, vp, vp, vp, vp, ci, vp, vp, vp,
                             ll, ll, ll, ll, ll, ci, vp, ci, vp, vp, vp, vp, vp, sz, ci]),
    "pk_mxfp8_scale_stride": (sz, [ci]),
    "pk_quantize_mxfp8": (ci, [vp, vp, vp, vp, ci, ci]),
    "pk_quantize_mxfp8_many": (ci, [vp, ci, vp, vp, vp, vp, vp]),
    "pk_query": (ci, [ctypes.POINTER(ci), ctypes.POINTER(ci), ctypes.POINTER(ci), ctypes.POINTER(ci),
                      ctypes.POINTER(sz)]),
    "prime_decode_status_string": (ctypes.c_char_p, [ci]),
    "pk_set_trace": (None, [vp]),
    "decode360": (ci, [vp, ci, vp, vp, vp, vp, vp, vp, ci, vp, vp, vp, ll, ll, ll, ll, ll, ci, vp, ci,
                       vp, vp, vp, sz, vp, sz, ci, ci]),
    "decode360_workspace_bytes": (sz, []),
    "decode360_debug_bytes": (sz, []),
    "decode360_status_string": (ctypes.c_char_p, [ci]),
    "mk_decode": (ci, [vp, ci, vp, ci, vp, vp, vp, ci, vp, vp, vp, vp, vp, ll, ll, ll, ll, ll, ci, vp,
                       ci, vp, vp, sz, ci]),
    "mk_workspace_bytes": (sz, [ci, ci]),
    "mk_status_string": (ctypes.c_char_p, [ci]),
    "block360_decode": (ci, [vp, ci, vp, vp, vp, vp, ci, vp, vp, vp, ll, ll, ll, ll, ll, ci, vp, ci, vp, vp, sz,
                             vp, sz, ci]),
    "block360_workspace_bytes": (sz, []),
    "block360_debug_bytes": (sz, []),
    "block360_status_string": (ctypes.c_char_p, [ci]),
    # include/prime_lossless.h
    "lossless_scan_workspace_bytes": (sz, []),
    "lossless_encode_layer": (ci, [vp, vp, vp, vp, vp, vp, vp, vp, sz, vp, ctypes.c_uint, vp]),
    "lossless_encode_workspace_bytes": (sz, [ci]),
    "lossless_encode_layers": (ci, [ci, vp, vp, vp, vp, vp, vp, vp, vp, vp, sz, vp]),
    "lossless_decode_layer": (ci, [vp, vp, vp, vp, vp]),
    "lossless_write_descriptor": (ci, [vp, ci, vp, vp, vp, vp, vp, vp]),
    "decode360_lossless": (ci, [vp, ci, vp, vp, vp, vp, vp, vp, ci, vp, vp, vp, ll, ll, ll, ll, ll, ci, vp, ci,
                                vp, vp, vp, sz, vp, sz, ci, ci, vp]),
    "pk_decode_lossless": (ci, [vp, ci, ci, ci, vp, ci, vp, vp, vp, vp, vp, ci, vp, vp, vp,
                                ll, ll, ll, ll, ll, ci, vp, ci, vp, vp, vp, vp, vp, sz, ci, vp]),
}


def library() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        if not LIB_PATH.is_file():
            raise RuntimeError(f"{LIB_PATH} is missing: build it with `python -m prime_kernels_amd.build`")
        lib = ctypes.CDLL(str(LIB_PATH))
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _lib = lib
    return _lib


def status_string(rc: int) -> str:
    return library().prime_decode_status_string(rc).decode()


def host_path(torch_version: str) -> Path:
    """The host module built against `torch_version` and this Python: its C++ interfaces are those of that
    torch alone, so the file's name says which."""
    return LIB_PATH.with_name(f"_host_step-torch{torch_version}.{sysconfig.get_config_var('SOABI')}.so")


def host():
    """The host module, make_spec and step (csrc/host_step.cpp), or None (with one warning) when there is
    no build of it for the running torch and Python: decode_step then checks in Python, for about 200 us
    more a call."""
    global _host
    if _host is None:
        import torch

        path = host_path(torch.__version__)
        if path.is_file():
            loader = importlib.machinery.ExtensionFileLoader("_host_step", str(path))
            module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_host_step", loader))
            loader.exec_module(module)
            _host = module
        else:
            warnings.warn(f"{path} is missing: decode_step checks its arguments in Python; build it with "
                          "`python -m prime_kernels_amd.build`", RuntimeWarning, stacklevel=2)
            _host = False
    return _host or None


def entry_address(name: str) -> int:
    """Address of a library entry point, for the host module."""
    return ctypes.cast(getattr(library(), name), ctypes.c_void_p).value
