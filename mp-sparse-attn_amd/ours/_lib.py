"""ctypes binding of libmpsa.so (the C ABI declared in include/mpsa.h).

PyTorch is used for device memory and streams only: tensors are handed over as raw device
pointers, sizes and element strides, and kernels are enqueued on torch's current stream.
"""

import ctypes
import importlib.machinery
import importlib.util
import os

import torch

BF16, F16, F32, F8E5M2 = 0, 1, 2, 3
FMT_E4M3, FMT_E5M2, FMT_E2M1 = 0, 1, 4
MODE_MXFP4, MODE_MXFP8, MODE_DIAG, MODE_ROUTED, MODE_MIXED = 0, 1, 2, 3, 4

# names of the MPSA_ATTN_* and MPSA_GEMM_* kernels
ATTN_KERNELS = {"auto": 0, "general": 1, "paired": 2, "short1": 3, "short2": 4, "short4": 5, "sequence": 6, "tile": 7}
GEMM_KERNELS = {"auto": 0, "general": 1, "split": 2, "tile128": 3, "tile256": 4,
                "split1x1": 11, "split1x2": 12, "split1x4": 14, "split2x2": 22, "split2x4": 24, "split4x4": 44}

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("MPSA_LIB_PATH") or os.path.join(os.path.dirname(_HERE), "lib", "libmpsa.so")

_i64, _int, _vp, _f32 = ctypes.c_int64, ctypes.c_int, ctypes.c_void_p, ctypes.c_float
_p64 = ctypes.POINTER(ctypes.c_int64)
_four = ctypes.c_int64 * 4


class AttnDesc(ctypes.Structure):
    """``mpsa_attn_desc`` of include/mpsa.h."""
    _fields_ = ([(n, _i64) for n in ("B", "Hq", "Hkv", "nq", "nk", "D")]
                + [(n, _i64 * 4) for n in ("q_strides", "k_strides", "v_strides", "o_strides")]
                + [(n, ctypes.c_int32) for n in ("dtype", "o_dtype", "tile", "causal", "mode", "fmt8", "smooth_k", "skip")]
                + [(n, _f32) for n in ("pre_scale_q", "skip_thresh", "route_thresh")])


class QuantizeJob(ctypes.Structure):
    """``mpsa_quantize_job`` of include/mpsa.h."""
    _fields_ = ([("x", _vp)] + [(n, _i64) for n in ("B", "H", "N", "D")] + [("x_strides", _i64 * 4), ("pre_scale", _f32), ("fmt", ctypes.c_int32), ("emax_elem", ctypes.c_int32),
                ("codes", _vp), ("scales", _vp), ("out_rows", _i64)])


# name -> (restype, argtypes); must list every symbol include/mpsa.h declares
SIGNATURES = {
    "mpsa_version": (_int, []),
    "mpsa_last_error": (ctypes.c_char_p, []),
    "mpsa_init": (_int, []),
    "mpsa_e2m1_encode": (_int, [_vp, _i64, _vp, _vp]),
    "mpsa_e2m1_decode": (_int, [_vp, _i64, _vp, _vp]),
    "mpsa_e8m0_encode": (_int, [_vp, _i64, _vp, _vp]),
    "mpsa_e8m0_decode": (_int, [_vp, _i64, _vp, _vp]),
    "mpsa_fp8_encode": (_int, [_vp, _i64, _int, _vp, _vp]),
    "mpsa_e2m1_pack": (_int, [_vp, _i64, _i64, _i64, _vp, _vp]),
    "mpsa_e2m1_pack_pair": (_int, [_vp, _i64, _i64, _vp] * 2 + [_vp]),
    "mpsa_e2m1_unpack": (_int, [_vp, _i64, _i64, _i64, _vp, _vp]),
    "mpsa_scales_to_5d": (_int, [_vp, _i64, _i64, _i64, _vp, _vp]),
    "mpsa_scales_from_5d": (_int, [_vp, _i64, _i64, _i64, _vp, _vp]),
    "mpsa_quantize_mx_as": (_int, [_vp, _int, _i64, _i64, _i64, _i64, _p64, _vp, _f32, _int, _int, _vp, _vp, _i64, _int, _int, _vp]),
    "mpsa_quantize_mx_pair": (_int, [ctypes.POINTER(QuantizeJob)] * 2 + [_int, _int, _int, _vp]),
    "mpsa_quantize_mx": (_int, [_vp, _int, _i64, _i64, _i64, _i64, _p64, _vp, _f32, _int, _int, _vp, _vp, _i64, _vp]),
    "mpsa_seq_mean_workspace": (_i64, [_i64, _i64, _i64, _i64]),
    "mpsa_seq_mean": (_int, [_vp, _int, _i64, _i64, _i64, _i64, _p64, _vp, _vp, _vp]),
    "mpsa_seq_mean_static": (_int, [_vp, _int, _i64, _i64, _i64, _i64, _p64, _vp, _vp]),
    "mpsa_quantize_mx_dual": (_int, [_vp, _int, _i64, _i64, _i64, _i64, _p64, _vp, _f32, _int, _int, _int,
                                     _vp, _vp, _vp, _vp, _i64, _vp]),
    "mpsa_gemm_mx": (_int, [_vp, _vp, _int, _vp, _vp, _int, _i64, _i64, _i64, _vp, _int, _i64, _vp]),
    "mpsa_gemm_mx_batched": (_int, [_vp, _vp, _int, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _vp, _int, _i64, _vp]),
    "mpsa_gemm_mx_packed": (_int, [_vp, _vp, _int, _vp, _vp, _int, _i64, _i64, _i64, _vp, _int, _i64, _vp]),
    "mpsa_gemm_mx_batched_packed": (_int, [_vp, _vp, _int, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _vp, _int, _i64, _vp]),
    "mpsa_gemm_mx_on": (_int, [_int, _vp, _vp, _int, _vp, _vp, _int, _int] + [_i64] * 6 + [_vp, _int, _i64, _vp]),
    "mpsa_gemm_kernel": (_int, [_int, _int, _int] + [_i64] * 5),
    "mpsa_v_tiles": (_int, [_vp, _int, _i64, _i64, _i64, _i64, _p64, _int, _vp, _vp]),
    "mpsa_attn_prepare": (_int, [_vp, _p64, _vp, _p64, _vp, _p64, _int, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _int,
                                 _f32, _vp] + [_vp] * 9 + [_vp]),
    "mpsa_attn_fwd": (_int, [_vp] * 8 + [_int, _vp, _int, _vp, _int, _p64,
                             _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _int, _vp]),
    "mpsa_attn_fwd_q16": (_int, [_vp, _p64, _int, _f32] + [_vp] * 4 + [_int, _vp, _int, _vp, _int, _p64,
                                 _i64, _i64, _i64, _i64, _i64, _int, _int, _int, _vp]),
    "mpsa_attn_kernel": (_int, [_int] + [_i64] * 6 + [_int, _int, _int]),
    "mpsa_attn_fwd_on": (_int, [_int] + [_vp] * 8 + [_int, _vp, _int, _vp, _int, _p64,
                                _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _int, _vp]),
    "mpsa_attn_fwd_q16_on": (_int, [_int, _vp, _p64, _int, _f32] + [_vp] * 4 + [_int, _vp, _int, _vp, _int, _p64,
                                    _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _int, _vp]),
    "mpsa_attn_fwd_q16_supported": (_int, [_i64, _i64, _i64, _i64, _i64, _int, _int, _int]),
    "mpsa_attn_fwd_skip": (_int, [_vp] * 8 + [_int, _vp, _int, _vp, _int, _p64,
                                  _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _int, _f32, _vp, _vp]),
    "mpsa_route_workspace": (_i64, [_i64, _i64, _i64, _i64, _i64, _i64, _int]),
    "mpsa_route_tiles": (_int, [_vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _f32, _f32, _vp, _vp, _vp, _vp, _vp]),
    "mpsa_skip_route_supported": (_int, [_i64, _i64, _i64, _int, _int, _int]),
    "mpsa_skip_route_workspace": (_i64, [_i64, _i64, _i64, _i64, _int]),
    "mpsa_skip_route": (_int, [_vp] * 8 + [_int, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _int, _f32, _vp, _vp, _vp, _vp, _vp, _vp]),
    "mpsa_attn_call_workspace": (_i64, [ctypes.POINTER(AttnDesc)]),
    "mpsa_attn_call": (_int, [ctypes.POINTER(AttnDesc)] + [_vp] * 7),
    "mpsa_attn_call_workspace_on": (_i64, [_int, ctypes.POINTER(AttnDesc)]),
    "mpsa_attn_call_on": (_int, [_int, ctypes.POINTER(AttnDesc)] + [_vp] * 7),
    "mpsa_attn_fwd_routed": (_int, [_vp] * 8 + [_int, _vp, _int, _vp, _int, _p64,
                                    _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _vp, _vp, _vp]),
}

_lib = None


class MpsaError(RuntimeError):
    """A libmpsa entry point returned a negative status."""

    def __init__(self, code, message):
        super().__init__(f"libmpsa error {code}: {message}")
        self.code = code


def lib():
    """Load libmpsa.so once.  Raises if it has not been built -- there is no fallback."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `python mp-sparse-attn_amd/build.py` "
                "(hipcc, gfx950). The MXFP path has no CPU or eager fallback.")
        handle = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = res
            fn.argtypes = args
        _lib = handle
        # set-up of the current device up front, so that even a caller's first launch there can be captured into a HIP
        # graph.  Other devices are set up by the entry points on their first use (mpsa_ensure_init); a caller that wants
        # to capture a first call on another device calls mpsa_init() with that device current.  (No device here means no
        # set-up: the entry points report their own errors.)
        if torch.cuda.is_available():
            status = handle.mpsa_init()
            if status != 0:
                raise MpsaError(status, handle.mpsa_last_error().decode("utf-8", "replace"))
    return _lib


_host = None


class _NoHost:
    """Stands in for the extension where MPSA_LIB_PATH names another library than the one it is linked to."""
    quantize = quantize_pair = pack_pair = matmul = matmul_batched = attention = staticmethod(lambda *args: None)


def host():
    """The native host side of short calls (csrc/host.cpp).  Its functions return None for anything but the usual case."""
    global _host
    if _host is None:
        lib()
        if os.environ.get("MPSA_LIB_PATH"):
            _host = _NoHost
            return _host
        path = os.path.join(os.path.dirname(LIB_PATH), "mpsa_host.so")
        if not os.path.exists(path):
            raise RuntimeError(f"{path} is missing: build it with `python mp-sparse-attn_amd/build.py`")
        loader = importlib.machinery.ExtensionFileLoader("mpsa_host", path)
        module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("mpsa_host", path, loader=loader))
        loader.exec_module(module)
        _host = module
    return _host


def check(status):
    if status != 0:
        raise MpsaError(status, lib().mpsa_last_error().decode("utf-8", "replace"))


_DTYPE_IDS = {torch.bfloat16: BF16, torch.float16: F16, torch.float32: F32, torch.float8_e5m2: F8E5M2}


def dtype_id(dtype):
    try:
        return _DTYPE_IDS[dtype]
    except KeyError:
        raise ValueError(f"unsupported dtype {dtype}") from None


def require_device(*tensors):
    for t in tensors:
        if not isinstance(t, torch.Tensor) or not t.is_cuda:
            raise RuntimeError("the MXFP path runs on HIP device tensors only (got a %s tensor); "
                               "there is no CPU fallback" % (t.device if isinstance(t, torch.Tensor) else type(t)))


def raw_stream(tensor):
    """:func:`stream_ptr` of a device tensor's device."""
    return torch._C._cuda_getCurrentRawStream(tensor.get_device())


def stream_ptr(device=None):
    """Handle of torch's current stream on a device (an int; 0 is the default stream).  The raw query takes a tenth of a
    microsecond, building a ``torch.cuda.Stream`` to read its handle two."""
    index = getattr(device, "index", None)
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)


def ptr(t):
    return t.data_ptr() if t is not None else None


class on_device:
    """``torch.cuda.device`` for the entry points: nothing but one query where the device is current already."""

    __slots__ = ("want", "before")

    def __init__(self, device):
        self.want = device.index

    def __enter__(self):
        self.before = torch._C._cuda_getDevice()
        if self.before != self.want:
            torch.cuda.set_device(self.want)

    def __exit__(self, *exc):
        if self.before != self.want:
            torch.cuda.set_device(self.before)
        return False


def strides4(t):
    assert t.dim() == 4
    return _four(*t.stride())
