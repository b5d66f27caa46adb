"""ctypes binding of libaf3_dpa.so (the C ABI declared in include/af3_dpa.h).

There is no fallback: if the library is missing, loading raises and every op fails loudly.
"""
import ctypes
import os
import warnings

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libaf3_dpa.so")
HOST_PATH = os.path.join(_HERE, "_host.so")

AF3_F32, AF3_BF16, AF3_FP8_E4M3, AF3_FP8_E5M2 = 0, 1, 2, 3
ABI_VERSION = 4
STATIC_SCRATCH_BYTES = 16 * 1024 * 1024   # AF3_STATIC_SCRATCH_BYTES

i64, i32, f32, vp = ctypes.c_int64, ctypes.c_int32, ctypes.c_float, ctypes.c_void_p


class DpaParams(ctypes.Structure):
    """Mirror of struct af3_dpa_params."""
    _fields_ = [
        ("q", vp), ("k", vp), ("v", vp), ("bias", vp), ("key_mask", vp), ("out", vp),
        ("B", i64), ("H", i64), ("L", i64), ("D", i64),
        ("q_stride", i64 * 3), ("k_stride", i64 * 3), ("v_stride", i64 * 3), ("out_stride", i64 * 3),
        ("bias_stride", i64 * 2), ("key_mask_stride_b", i64),
        ("io_dtype", i32), ("bias_dtype", i32), ("out_dtype", i32), ("mma_dtype", i32),
        ("softmax_scale", f32), ("q_descale", f32), ("k_descale", f32), ("v_descale", f32),
        ("force_generic", i32), ("reserved", i32),
        ("device_descales", vp),
        ("workspace", vp), ("workspace_bytes", i64),
        ("q_lo", vp), ("k_lo", vp),
        ("gate", vp), ("gate_stride", i64 * 3),
    ]


class GridAttentionParams(ctypes.Structure):
    """Mirror of struct af3_grid_attention_params."""
    _fields_ = [
        ("pair", vp), ("pair_stride", i64 * 2),
        ("q_proj", vp), ("k_proj", vp), ("v_proj", vp), ("gating_query", vp),
        ("bias", vp), ("bias_stride", i64 * 2), ("bias_dtype", i32), ("dtype", i32),
        ("key_mask", vp), ("key_mask_stride_b", i64),
        ("out", vp), ("out_stride", i64 * 2),
        ("B", i64), ("N", i64), ("C", i64), ("head", i64),
        ("workspace", vp), ("workspace_bytes", i64),
    ]


QKV_SCRATCH_FLOATS = 768   # AF3_QKV_SCRATCH_FLOATS

# name -> (restype, argtypes); every symbol include/af3_dpa.h declares
SYMBOLS = {
    "af3_dpa_forward": (ctypes.c_int, [ctypes.POINTER(DpaParams), vp]),
    "af3_dpa_forward_static_scratch": (ctypes.c_int, [ctypes.POINTER(DpaParams), vp]),
    "af3_dpa_select_kernel": (ctypes.c_int, [ctypes.POINTER(DpaParams)]),
    "af3_dpa_workspace_bytes": (ctypes.c_int64, [ctypes.POINTER(DpaParams)]),
    "af3_grid_attention_forward": (ctypes.c_int, [ctypes.POINTER(GridAttentionParams), vp]),
    "af3_grid_attention_workspace_bytes": (ctypes.c_int64, [ctypes.POINTER(GridAttentionParams)]),
    "af3_grid_attention_supported": (ctypes.c_int, [ctypes.POINTER(GridAttentionParams)]),
    "af3_layernorm_pair_bias": (ctypes.c_int, [vp, ctypes.POINTER(i64), vp, vp, f32, vp, vp, vp, ctypes.POINTER(i64), i64, i64, i64, i64, i32, vp]),
    "af3_gated_linear_unit": (ctypes.c_int, [vp, vp, vp, i64, i64, i64, i32, vp]),
    "af3_silu_mul": (ctypes.c_int, [vp, vp, i64, i64, i32, vp]),
    "af3_linear": (ctypes.c_int, [vp, vp, vp, i64, i64, i64, i32, vp]),
    "af3_convert": (ctypes.c_int, [vp, i32, vp, i32, i64, vp]),
    "af3_amax": (ctypes.c_int, [vp, i32, i64, vp, vp]),
    "af3_quantize_fp8_e4m3": (ctypes.c_int, [vp, i32, vp, i64, i64, i64, i32, i64, i64, f32, vp, vp, vp, vp]),
    "af3_quantize_qkv_fp8_e4m3": (ctypes.c_int, [vp, vp, vp, i32, i64, i64, i64, i64, f32, vp, vp, vp, i64, vp, vp, vp, vp, vp]),
    "af3_pad_nd": (ctypes.c_int, [vp, vp, i32, ctypes.POINTER(i64), ctypes.POINTER(i64), ctypes.POINTER(i64), i32, ctypes.c_uint32, vp]),
    "af3_vnni_repack_bf16": (ctypes.c_int, [vp, vp, i64, i64, i64, vp]),
    "af3_status_string": (ctypes.c_char_p, [ctypes.c_int]),
    "af3_abi_version": (ctypes.c_int, []),
}

# ... and those that only this package's two host sides call (not part of the ABI)
INTERNAL_SYMBOLS = {
    "af3_project_suits": (ctypes.c_int, [i64, i64, i64]),
    "af3_project": (ctypes.c_int, [vp, vp, vp, vp, i64, i64, i64, i32, vp]),
}

_lib = None


def load():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(
                f"{LIB_PATH} is missing: build it with `python -m af3_kernels_amd.build` (hipcc, gfx950). "
                "There is no CPU or PyTorch fallback for these ops.")
        lib = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in (SYMBOLS | INTERNAL_SYMBOLS).items():
            fn = getattr(lib, name)
            fn.restype, fn.argtypes = res, args
        if lib.af3_abi_version() != ABI_VERSION:
            raise ImportError(f"{LIB_PATH} has ABI version {lib.af3_abi_version()}, this package expects {ABI_VERSION}: rebuild it")
        _lib = lib
    return _lib


class _Host:
    """The native host side of the entry points (csrc/host.cpp), looked for when it is first needed: a package that is built after
    its import works from then on.  While `_host.so` alone is missing every call is answered None, which sends it to the Python
    implementation (a warning says so, once); without the kernels' library a call raises, as load() does."""
    FUSED_WEIGHT, Q_BIAS_ROW, OUT_PROJ_T, GLU_T = 1, 2, 3, 4   # as in host.cpp
    _warned = False

    def __getattr__(self, name):   # (reached until the module's functions are in this object)
        load()
        if os.path.exists(HOST_PATH):
            import torch  # noqa: F401 -- its libraries must be loaded first
            from . import _host
            self.__dict__.update((k, v) for k, v in vars(_host).items() if not k.startswith("__"))
            return getattr(_host, name)
        if not _Host._warned:
            _Host._warned = True
            warnings.warn(f"{HOST_PATH} is missing: calls are prepared in Python, which takes 10 to 40 us more each; build it with `python -m af3_kernels_amd.build`", RuntimeWarning)
        return lambda *args: None


def load_host():
    """The native host side where it is built already (its functions are then the module's own), else a stand-in that finds it later."""
    if not (os.path.exists(HOST_PATH) and os.path.exists(LIB_PATH)):
        return _Host()
    load()
    import torch  # noqa: F401 -- its libraries must be loaded first
    from . import _host
    return _host


def check(status: int, what: str):
    if status != 0:
        msg = load().af3_status_string(status).decode()
        exc = ValueError if status in (-2, -3, -4, -5, -7, -9) else RuntimeError
        raise exc(f"{what}: {msg} (af3_status {status})")
