"""ctypes binding of libpackkv_hip.so (the C ABI declared in include/packkv.h).

The library is the product: there is no fallback.  If it has not been built, or cannot be
loaded, importing the op surface fails with instructions instead of silently running
something else.
"""
import ctypes
import os
import warnings

_HERE = os.path.dirname(os.path.abspath(__file__))
# PACKKV_HIP_LIB names another build of the same library (kernel development: A/B runs of two builds)
LIB_PATH = os.environ.get("PACKKV_HIP_LIB") or os.path.join(_HERE, "libpackkv_hip.so")
HOST_SYMBOLS = ("pkv_attn_decode", "pkv_window_append", "pkv_dense_view", "pkv_kq_mat_vec_mul", "pkv_wv_mat_vec_mul", "pkv_fused_kq",
                "pkv_fused_wv")

F16, BF16 = 0, 1
OK, ERR_UNSUPPORTED, ERR_INVALID, ERR_HIP, ERR_CAPACITY, ERR_INTERNAL = range(6)
ATTN_REF_ROUNDING, ATTN_OUT_F32 = 1, 2

_vp = ctypes.c_void_p
_i = ctypes.c_int
_u64 = ctypes.c_uint64
_i64 = ctypes.c_int64
_f = ctypes.c_float
_fp = ctypes.POINTER(ctypes.c_float)
_u64p = ctypes.POINTER(ctypes.c_uint64)


class AttnArgs(ctypes.Structure):
    _fields_ = [
        ("k_stream", _vp), ("k_info", _vp), ("v_stream", _vp), ("v_info", _vp),
        ("k_bytes", _u64), ("v_bytes", _u64),
        ("k_scale", _vp), ("k_zero", _vp), ("v_scale", _vp), ("v_zero", _vp),
        ("q", _vp), ("out", _vp), ("k_win", _vp), ("v_win", _vp),
        ("B", _i), ("Hq", _i), ("Hkv", _i), ("T_c", _i), ("T_w", _i),
        ("k_bits", _i), ("v_bits", _i), ("dtype", _i), ("sm_scale", _f), ("variant", _i),
        ("par_stride", _i), ("win_stride", _i), ("flags", _i),
    ]


class AppendSide(ctypes.Structure):
    _fields_ = [("x", _vp), ("stride_b", _i64), ("stride_h", _i64), ("stride_t", _i64), ("stream", _vp), ("capacity", _u64),
                ("used", _u64), ("info_tail", _vp), ("scale_tail", _vp), ("zero_tail", _vp), ("rel", _f), ("bits", _i),
                ("cos", _vp), ("sin", _vp), ("rot_stride_b", _i64)]


class CutArgs(ctypes.Structure):
    _fields_ = ([(n, _vp) for n in ("k_new", "v_new", "cos", "sin")] +
                [(n, _i64) for n in ("stride_b", "stride_h", "stride_t", "rot_stride_b")] +
                [(n, _vp) for n in ("k_pend", "v_pend", "k_win", "v_win", "k_stage", "v_stage", "k_pend_out", "v_pend_out",
                                    "k_win_out", "v_win_out")] +
                [(n, _i) for n in ("dtype", "B", "H", "n", "pend", "buf", "stage", "pend_out", "win_stride")] +
                [("k_rel", _f), ("v_rel", _f)])


# name -> (restype, argtypes); every symbol include/packkv.h declares
SIGNATURES = {
    "pkv_abi_version": (_i, []),
    "pkv_last_error": (ctypes.c_char_p, []),
    "pkv_block_bound": (_u64, [_i, _i, _i, _i]),
    "pkv_k_encode": (_i, [_vp, _vp, _u64, _vp, _i, _i, _i, _i, _i, _u64p, _fp, _vp]),
    "pkv_v_encode": (_i, [_vp, _vp, _u64, _vp, _i, _i, _i, _i, _i, _u64p, _fp, _vp]),
    "pkv_encode_status": (_i, [_vp, _i, _u64p]),
    "pkv_k_encode_p": (_i, [_vp, _vp, _u64, _vp, _i, _i, _i, _i, _u64p, _fp, _vp]),
    "pkv_v_encode_p": (_i, [_vp, _vp, _u64, _vp, _i, _i, _i, _i, _u64p, _fp, _vp]),
    "pkv_k_decode_p": (_i, [_vp, _u64, _vp, _vp, _i, _i, _i, _i, _fp, _vp]),
    "pkv_v_decode_p": (_i, [_vp, _u64, _vp, _vp, _i, _i, _i, _i, _fp, _vp]),
    "pkv_block_bound_p": (_u64, [_i, _i]),
    "pkv_k_decode": (_i, [_vp, _u64, _vp, _vp, _i, _i, _i, _i, _i, _fp, _vp]),
    "pkv_v_decode": (_i, [_vp, _u64, _vp, _vp, _i, _i, _i, _i, _i, _fp, _vp]),
    "pkv_quant_params": (_i, [_vp, _i, _i, _i, _i, _f, _vp, _vp, _fp, _vp]),
    "pkv_quant_codes": (_i, [_vp, _vp, _i, _i, _i, _i, _f, _f, _vp, _vp, _vp, _vp, _vp, _vp, _vp]),
    "pkv_quantize": (_i, [_vp, _i, _i, _i, _i, _vp, _vp, _vp, _vp, _fp, _vp]),
    "pkv_dequantize": (_i, [_vp, _i, _i, _i, _i, _vp, _vp, _vp, _fp, _vp]),
    "pkv_median_order": (_i, [_vp, _i, _i, _i, _i, _f, _i, _i, _vp, _vp, _vp, _fp, _vp]),
    "pkv_k_quant_encode_perm": (_i, [_vp, _i, _i, _i, _i, _f, _i, _vp, _i, _vp, _u64, _vp, _vp, _vp, _u64p, _fp, _vp]),
    "pkv_v_quant_encode_perm": (_i, [_vp, _i, _i, _i, _i, _f, _i, _vp, _i, _vp, _vp, _vp, _u64, _vp, _vp, _vp, _u64p, _fp, _vp]),
    "pkv_k_quant_encode": (_i, [_vp, _i, _i, _i, _i, _f, _i, _vp, _u64, _vp, _vp, _vp, _u64p, _fp, _vp]),
    "pkv_v_quant_encode": (_i, [_vp, _i, _i, _i, _i, _f, _i, _vp, _u64, _vp, _vp, _vp, _u64p, _fp, _vp]),
    "pkv_k_quant_encode_append": (_i, [_vp, _i, _i, _i, _i, _f, _i, _vp, _u64, _u64, _vp, _vp, _vp, _i, _u64p, _fp, _vp]),
    "pkv_v_quant_encode_append": (_i, [_vp, _i, _i, _i, _i, _f, _i, _vp, _u64, _u64, _vp, _vp, _vp, _i, _u64p, _fp, _vp]),
    "pkv_kv_quant_encode_append": (_i, [ctypes.POINTER(AppendSide), ctypes.POINTER(AppendSide), _i, _i, _i, _i, _i, _u64p, _u64p, _vp]),
    "pkv_kv_quant_encode_alone": (_i, [ctypes.POINTER(AppendSide), ctypes.POINTER(AppendSide), _i, _i, _i, _i, _i, _vp, _i, _u64p, _u64p, _vp]),
    "pkv_kv_quant_encode_perm": (_i, [ctypes.POINTER(AppendSide), ctypes.POINTER(AppendSide), _i, _i, _i, _i, _vp, _i, _vp, _vp, _u64p, _u64p, _vp]),
    "pkv_window_cut": (_i, [ctypes.POINTER(CutArgs), _vp]),
    "pkv_window_append": (_i, [_vp, _vp, _vp, _vp, _i, _i, _i, _i, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64,
                               ctypes.c_int64, _vp, _vp, _i, _i, _vp]),
    "pkv_bit_pack_size": (_i, [_vp, _i, _i, _i, _u64p, ctypes.POINTER(ctypes.c_uint32), _fp, _vp]),
    "pkv_bit_pack_size_pair": (_i, [_vp, _vp, _vp, _i, _i, _i, _i, _u64p, ctypes.POINTER(ctypes.c_uint32), _vp]),
    "pkv_median_repack": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _fp, _vp]),
    "pkv_greedy_repack": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _fp, _vp]),
    "pkv_kq_mat_vec_mul": (_i, [_vp, _u64, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _fp, _vp]),
    "pkv_wv_mat_vec_mul": (_i, [_vp, _u64, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _fp, _vp]),
    "pkv_fused_kq": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _fp, _vp]),
    "pkv_fused_wv": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _fp, _vp]),
    "pkv_attn_decode": (_i, [ctypes.POINTER(AttnArgs), _fp, _vp]),
    "pkv_attn_decode_noalloc": (_i, [ctypes.POINTER(AttnArgs), _vp]),
    "pkv_dense_view": (_i, [ctypes.POINTER(AttnArgs), _vp, _vp, _vp]),
    "pkv_stream_release": (_i, [_vp]),
}

_lib = None
host = None        # the native host side of the repeated calls (csrc/pkv_host.cpp), or NO_HOST, once the library is loaded


class PackKVError(RuntimeError):
    """A C-ABI call returned a non-zero status; ``code`` holds the PKV_ERR_* value."""

    def __init__(self, code, message):
        super().__init__(message)
        self.code = code


class _NoHost:
    """Serves no call: the general code of ops.py does them all."""

    def __getattr__(self, name):
        return lambda *args: None


NO_HOST = _NoHost()


def _load_host(lib):
    """The native host side; NO_HOST, with a warning, where it is missing or was built for another torch (the library itself
    knows nothing of torch, and the general code needs nothing but it)."""
    import torch
    try:
        from . import _host
        made_for = getattr(_host, "torch", "unknown")
        why = None if made_for == torch.__version__ else "built for torch %s, this is %s" % (made_for, torch.__version__)
    except ImportError as e:
        why = str(e)
    if why:
        warnings.warn("packkv_amd._host is not used (%s): the calls that a decode loop repeats take 4 to 8 us more of host time each. "
                      "`python -m packkv_amd.build` makes it." % why, RuntimeWarning, stacklevel=3)
        return NO_HOST
    _host.bind(*(ctypes.cast(getattr(lib, name), _vp).value for name in HOST_SYMBOLS))
    return _host


def load():
    """Load the library once and attach prototypes.  Raises ImportError when it is missing."""
    global _lib, host
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            "libpackkv_hip.so is not built (%s). Build it with `python -m packkv_amd.build` "
            "(needs hipcc, targets gfx950); there is no CPU fallback." % LIB_PATH)
    try:
        lib = ctypes.CDLL(LIB_PATH)
    except OSError as e:  # pragma: no cover - depends on the machine
        raise ImportError("cannot load %s: %s" % (LIB_PATH, e))
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    host, _lib = _load_host(lib), lib
    return lib


def check(rc):
    if rc != 0:
        msg = load().pkv_last_error().decode("utf-8", "replace")
        raise PackKVError(rc, msg or ("packkv error %d" % rc))
