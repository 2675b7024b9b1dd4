"""Loader of the HIP library behind the C ABI (include/sru_amd.h).

There is no fallback: if libsru_amd.so is missing or cannot be loaded, every
entry point of this package raises. The library is built in-tree by
`python -m sru_amd.build` (hipcc --offload-arch=gfx950).
"""
import ctypes
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libsru_amd.so")
ABI_VERSION = 8
STATE_INTERVAL = 8   # SRU_AMD_STATE_INTERVAL
STATIC_MAX_COLUMNS = 262144   # SRU_AMD_STATIC_MAX_COLUMNS
NORM_MAX_FEATURES = 4096       # SRU_AMD_NORM_MAX_FEATURES

F32, F16, BF16, F64 = 0, 1, 2, 3
X_AS_STREAMS, X_F32 = 0, 1   # SRU_AMD_X_AS_STREAMS, SRU_AMD_X_F32
LAYER_STEP, LAYER_ROWS = 1, 2      # what sru_amd_layer_route answers
# SRU_AMD_SMALL_*: small tensors held in the stream type
SMALL_WEIGHT_C, SMALL_BIAS, SMALL_INIT, SMALL_MASK, SMALL_SCALE, SMALL_LAST = 1, 2, 4, 8, 16, 32


class Shape(ctypes.Structure):
    """struct sru_amd_shape."""
    _fields_ = [
        ("length", ctypes.c_int64),
        ("batch", ctypes.c_int64),
        ("hidden", ctypes.c_int64),
        ("dirs", ctypes.c_int32),
        ("k", ctypes.c_int32),
        ("activation_type", ctypes.c_int32),
        ("skip_type", ctypes.c_int32),
        ("is_custom", ctypes.c_int32),
        ("dtype", ctypes.c_int32),
        ("state_interval", ctypes.c_int32),
        ("x_dtype", ctypes.c_int32),
    ]


_P = ctypes.c_void_p
SIGNATURES = {
    # name: (restype, argtypes) exactly as declared in include/sru_amd.h
    "sru_amd_forward": (ctypes.c_int, [ctypes.POINTER(Shape)] + [_P] * 12),
    "sru_amd_forward_small": (ctypes.c_int, [ctypes.POINTER(Shape), ctypes.c_uint32] + [_P] * 12),
    "sru_amd_state_bytes": (ctypes.c_size_t, [ctypes.POINTER(Shape)]),
    "sru_amd_backward_workspace_bytes": (ctypes.c_size_t, [ctypes.POINTER(Shape)]),
    "sru_amd_backward": (ctypes.c_int, [ctypes.POINTER(Shape)] + [_P] * 17 + [ctypes.c_size_t, _P]),
    "sru_amd_backward_small": (ctypes.c_int, [ctypes.POINTER(Shape), ctypes.c_uint32] + [_P] * 17 + [ctypes.c_size_t, _P]),
    "sru_amd_backward_static": (ctypes.c_int, [ctypes.POINTER(Shape)] + [_P] * 17),
    "sru_amd_layer_route": (ctypes.c_int, [ctypes.POINTER(Shape), ctypes.c_int64, ctypes.c_int64]),
    "sru_amd_layer_forward": (ctypes.c_int, [ctypes.POINTER(Shape), ctypes.c_uint32, ctypes.c_int64, ctypes.c_int64] + [_P] * 13),
    "sru_amd_stack_workspace_bytes": (ctypes.c_size_t, [ctypes.POINTER(Shape), ctypes.c_int64, ctypes.c_int64]),
    "sru_amd_stack_wanted_in_graph": (ctypes.c_int, [ctypes.POINTER(Shape), ctypes.c_int64, ctypes.c_int64]),
    "sru_amd_stack_forward": (ctypes.c_int, [ctypes.POINTER(Shape), ctypes.c_uint32, ctypes.c_int64, ctypes.c_int64] + [_P] * 11 + [ctypes.c_size_t, _P]),
    "sru_amd_product_wanted": (ctypes.c_int, [ctypes.c_int32] + [ctypes.c_int64] * 3),
    "sru_amd_product": (ctypes.c_int, [ctypes.c_int32] + [ctypes.c_int64] * 3 + [_P] * 4),
    "sru_amd_product_grad_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int32] + [ctypes.c_int64] * 3),
    "sru_amd_product_grad": (ctypes.c_int, [ctypes.c_int32] + [ctypes.c_int64] * 3 + [_P, _P, ctypes.c_int32, _P, _P, ctypes.c_size_t, _P]),
    "sru_amd_layer_norm_forward": (ctypes.c_int, [ctypes.c_int64, ctypes.c_int64, _P, ctypes.c_int, _P, _P,
                                                  ctypes.c_float, _P, ctypes.c_int, _P, _P, _P]),
    "sru_amd_layer_norm_backward_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int64, ctypes.c_int64]),
    "sru_amd_layer_norm_backward": (ctypes.c_int, [ctypes.c_int64, ctypes.c_int64, _P, ctypes.c_int, _P, _P, _P, _P,
                                                   ctypes.c_int, _P, _P, _P, _P, ctypes.c_size_t, _P]),
    "sru_amd_status_string": (ctypes.c_char_p, [ctypes.c_int]),
    "sru_amd_abi_version": (ctypes.c_int, []),
}

_lib = None


class LibraryError(RuntimeError):
    pass


def load():
    """Returns the loaded library with argument types set; raises LibraryError."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise LibraryError(
            f"{LIB_PATH} is missing: build it with `python -m sru_amd.build` "
            "(there is no fallback path for the SRU recurrence)")
    try:
        lib = ctypes.CDLL(LIB_PATH)
    except OSError as exc:
        raise LibraryError(f"cannot load {LIB_PATH}: {exc}") from exc
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    if lib.sru_amd_abi_version() != ABI_VERSION:
        raise LibraryError(f"{LIB_PATH} has ABI version {lib.sru_amd_abi_version()}, "
                           f"this package needs {ABI_VERSION}; rebuild it")
    _lib = lib
    return lib


_host = None


class GeneralHost:
    """Stands for the native host code where that cannot be used: nothing is plain, every call goes the
    general way of functional.py."""
    scan_forward = scan_backward = product = stack_forward = recurrence = layer = staticmethod(lambda *args: None)
    autocast_operand = staticmethod(lambda t: None)
    layer_forward = staticmethod(lambda *args: False)

    @staticmethod
    def observed():
        import torch
        return torch._C._len_torch_function_stack() > 0 or torch._C._len_torch_dispatch_stack() > 0


def host():
    """The native host code (csrc/host.cpp): calls in the plain case, from torch tensors to the C ABI. It
    is built against one release of torch and used with that one only; without it the same kernels run
    with more host time per call, after one warning."""
    global _host
    if _host is None:
        load()      # the library it calls, and the error where that is missing
        import torch
        try:
            from . import _host as module
            reason = None if module.torch_version == torch.__version__ else f"built for torch {module.torch_version}, not {torch.__version__}"
        except (ImportError, AttributeError) as exc:
            reason = str(exc)
        if reason:
            import warnings
            warnings.warn(f"sru_amd/_host.so cannot be used ({reason}): calls cost more host time; rebuild it with `python -m sru_amd.build`",
                          RuntimeWarning, stacklevel=2)
            module = GeneralHost
        _host = module
    return _host


def status_string(code):
    return load().sru_amd_status_string(code).decode()


def check(code, what):
    """Maps a non-zero status to the exception a caller of the reference would see:
    shape / flag problems are ValueError, everything else RuntimeError."""
    if code == 0:
        return
    msg = f"{what}: {status_string(code)} (sru_amd status {code})"
    if code in (2, 3, 4):
        raise ValueError(msg)
    raise RuntimeError(msg)
