"""ctypes binding of libkvq.so (include/kvq.h), and the native host path over it
(`host`, csrc/host.cpp).

Loading the library needs the ROCm runtime (libamdhip64) but no GPU; every argument
check in the library runs before any HIP call. There is deliberately no fallback: if the
library is missing the import of the op fails loudly.
"""
import ctypes
import importlib
import os
import warnings

_PKG_DIR = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_PKG_DIR, "libkvq.so")

# The native host path: each function returns None for a call it does not take, which then
# goes through the Python path. Until `lib` has loaded both libraries it takes none.
HOST_PATH = os.path.join(_PKG_DIR, "_host.so")


class _NoHost:
    @staticmethod
    def decode(*args):
        return None

    quantize = quantize_append = append_kv = reshape_and_cache = set_cu_count = decode


host = _NoHost
_cu_counts = {}  # compute units by device index, as the native path has been told


def __getattr__(name):
    if name == "HOST_BUILT":  # asked each time: a build may come after the import
        return os.path.exists(HOST_PATH)
    raise AttributeError(f"module {__name__!r} has no attribute {name!r}")


# kvq_status (include/kvq.h)
KVQ_OK = 0
KVQ_ERR_NULL_POINTER = -1
KVQ_ERR_SHAPE = -2
KVQ_ERR_UNSUPPORTED = -3
KVQ_ERR_ALIGNMENT = -4
KVQ_ERR_SPLITS = -5
KVQ_ERR_FORMAT = -6
KVQ_ERR_HIP = -7
KVQ_ERR_SCRATCH = -8

# KVQ_STATIC_SCRATCH_BYTES: the static device buffer of kvq_paged_decode_static
STATIC_SCRATCH_BYTES = 16 * 1024 * 1024

# kvq_kv_format
KV_FORMATS = {"fp16": 0, "int8": 1, "fp8_e4m3": 2, "int4": 3}

# Every symbol include/kvq.h declares; tests check the library exports all of them.
EXPORTED_SYMBOLS = (
    "kvq_version",
    "kvq_cache_format_version",
    "kvq_head_blocks",
    "kvq_status_string",
    "kvq_choose_num_splits",
    "kvq_plan_decode",
    "kvq_normalize_splits",
    "kvq_decode_split",
    "kvq_decode_merge",
    "kvq_decode_single",
    "kvq_paged_decode",
    "kvq_decode_units",
    "kvq_decode_units_split",
    "kvq_decode_units_merge",
    "kvq_plan_units",
    "kvq_quantize_cache",
    "kvq_quantize_append",
    "kvq_append_kv",
    "kvq_reshape_and_cache",
    "kvq_paged_decode_static",
)

_i32 = ctypes.c_int32
_i64 = ctypes.c_int64
_vp = ctypes.c_void_p
_fp = ctypes.POINTER(ctypes.c_float)


class DecodeArgs(ctypes.Structure):
    """Mirror of struct kvq_decode_args."""
    _fields_ = [
        ("q", _vp), ("q_stride_b", _i64), ("q_stride_h", _i64),
        ("k_cache", _vp), ("k_stride_blk", _i64), ("k_stride_tok", _i64), ("k_stride_head", _i64),
        ("v_cache", _vp), ("v_stride_blk", _i64), ("v_stride_tok", _i64), ("v_stride_head", _i64),
        ("block_table", _vp), ("bt_stride_b", _i64),
        ("seq_lens", _vp),
        ("out", _vp), ("o_stride_b", _i64), ("o_stride_h", _i64),
        ("batch", _i32), ("q_heads", _i32), ("kv_heads", _i32), ("head_dim", _i32),
        ("block_size", _i32), ("max_blocks", _i32), ("num_blocks", _i32),
        ("scale", ctypes.c_float),
        ("kv_format", _i32),
        ("k_group", _i32),
        ("k_scale", _vp), ("k_zero", _vp), ("v_scale", _vp), ("v_zero", _vp),
        ("waves_per_group", _i32),
        ("pipeline", _i32),
    ]


class KvqError(RuntimeError):
    """A libkvq call returned a negative kvq_status."""

    def __init__(self, func, status, text):
        super().__init__(f"{func} failed: {text} (status {status})")
        self.status = status


_lib = None


def lib():
    """The loaded library (loaded on first use)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(
                f"{LIB_PATH} is not built; run `python -m kvq_decode_amd.build` "
                "(there is no CPU fallback for this op)")
        L = ctypes.CDLL(LIB_PATH)
        L.kvq_version.restype = ctypes.c_char_p
        L.kvq_version.argtypes = []
        L.kvq_cache_format_version.restype = ctypes.c_int
        L.kvq_cache_format_version.argtypes = []
        L.kvq_head_blocks.restype = ctypes.c_int
        L.kvq_head_blocks.argtypes = [_i32, _i32]
        L.kvq_status_string.restype = ctypes.c_char_p
        L.kvq_status_string.argtypes = [ctypes.c_int]
        L.kvq_choose_num_splits.restype = ctypes.c_int
        L.kvq_choose_num_splits.argtypes = [_i32] * 7
        L.kvq_plan_decode.restype = ctypes.c_int
        L.kvq_plan_decode.argtypes = [_i32] * 8 + [ctypes.POINTER(_i32)] * 2
        L.kvq_plan_units.restype = ctypes.c_int
        L.kvq_plan_units.argtypes = [_i32] * 8 + [ctypes.POINTER(_i32)] * 2
        L.kvq_normalize_splits.restype = ctypes.c_int
        L.kvq_normalize_splits.argtypes = [_i32, _i32, ctypes.POINTER(_i32), ctypes.POINTER(_i32)]
        args_p = ctypes.POINTER(DecodeArgs)
        L.kvq_decode_split.restype = ctypes.c_int
        L.kvq_decode_split.argtypes = [args_p, _i32, _i32, _vp, _vp, _vp]
        L.kvq_decode_merge.restype = ctypes.c_int
        L.kvq_decode_merge.argtypes = [_vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _i32, _vp]
        L.kvq_decode_single.restype = ctypes.c_int
        L.kvq_decode_single.argtypes = [args_p, _vp]
        L.kvq_paged_decode.restype = ctypes.c_int
        L.kvq_paged_decode.argtypes = [args_p, _i32, _vp, _vp, _vp]
        L.kvq_decode_units.restype = ctypes.c_int
        L.kvq_decode_units.argtypes = [args_p, _i32, _vp, _vp, _vp]
        L.kvq_decode_units_split.restype = ctypes.c_int
        L.kvq_decode_units_split.argtypes = [args_p, _i32, _vp, _vp, _vp]
        L.kvq_decode_units_merge.restype = ctypes.c_int
        L.kvq_decode_units_merge.argtypes = [args_p, _i32, _vp, _vp, _vp]
        L.kvq_quantize_cache.restype = ctypes.c_int
        L.kvq_quantize_cache.argtypes = [args_p, _vp, _vp, _i64, _i64, _i64, _vp]
        L.kvq_quantize_append.restype = ctypes.c_int
        L.kvq_quantize_append.argtypes = [args_p, _vp, _vp, _vp, _vp]
        L.kvq_append_kv.restype = ctypes.c_int
        L.kvq_append_kv.argtypes = [args_p, _vp, _vp, _vp]
        L.kvq_reshape_and_cache.restype = ctypes.c_int
        L.kvq_reshape_and_cache.argtypes = [args_p, _vp, _vp, _i64, _i64, _vp, _i32, _vp]
        L.kvq_paged_decode_static.restype = ctypes.c_int
        L.kvq_paged_decode_static.argtypes = [args_p, _i32, _i32, _vp]
        _lib = L
        _load_host(L)
    return _lib


# libkvq.so's functions the native host path calls, in csrc/host.cpp's order
HOST_SYMBOLS = ("kvq_head_blocks", "kvq_plan_decode", "kvq_plan_units", "kvq_normalize_splits",
                "kvq_paged_decode", "kvq_decode_units", "kvq_quantize_cache",
                "kvq_quantize_append", "kvq_append_kv", "kvq_reshape_and_cache")


def _load_host(L):
    """Imports the native host path and binds it to the loaded library. It is loaded with the
    library and not with the package, so that a build run from a process that has imported the
    package is followed by the modules it built. The Python path is complete without it: one
    that is missing or fails to load costs host time only, and is reported as a warning."""
    global host
    try:
        import torch  # noqa: F401  (the module links against torch's libraries)
        importlib.invalidate_caches()
        module = importlib.import_module("kvq_decode_amd._host")
        bind_host(L, module)
    except Exception as e:
        why = "is not built" if not os.path.exists(HOST_PATH) else f"does not load ({e})"
        warnings.warn(f"{HOST_PATH} {why}: calls take the slower Python host path; run "
                      "`python -m kvq_decode_amd.build`", RuntimeWarning, stacklevel=3)
        return
    host = module
    for device, count in _cu_counts.items():
        host.set_cu_count(device, count)


def bind_host(L, module=None):
    """Points the native host path at the loaded library's functions."""
    (module or host).bind(check, *(ctypes.cast(getattr(L, name), _vp).value for name in HOST_SYMBOLS))


def set_cu_count(device, count):
    """Tells the native host path a device's compute units, now or once it is loaded."""
    _cu_counts[device] = count
    host.set_cu_count(device, count)


def check(func, status):
    """Raise KvqError for a negative status; return the status otherwise."""
    if status < 0:
        text = lib().kvq_status_string(status).decode()
        raise KvqError(func, status, text)
    return status


def version():
    return lib().kvq_version().decode()
