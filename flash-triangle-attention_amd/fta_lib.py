"""ctypes binding of libfta.so (see include/fta.h).  No torch types cross this boundary."""
from __future__ import annotations

import ctypes
import importlib.util
import os
import warnings

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libfta.so")
NATIVE_PATH = os.path.join(HERE, "fta_native.so")
MAX_L2 = 4096  # FTA_MAX_L2 of include/fta.h
STATIC_WORKSPACE_BYTES = 128 * 1024 * 1024  # FTA_STATIC_WORKSPACE_BYTES of include/fta.h


class Tensor5(ctypes.Structure):
    _fields_ = [("ptr", ctypes.c_void_p), ("stride", ctypes.c_int64 * 4)]


class Tensor4(ctypes.Structure):
    _fields_ = [("ptr", ctypes.c_void_p), ("stride", ctypes.c_int64 * 3)]


class Options(ctypes.Structure):
    _fields_ = [("dtype", ctypes.c_int), ("dbias_f32", ctypes.c_int), ("dropout_p", ctypes.c_float), ("seed", ctypes.c_uint64),
                ("precise", ctypes.c_int)]


_WEIGHTS = [(n, ctypes.c_void_p) for n in ("norm_weight", "norm_bias", "wq", "wk", "wv", "wb", "wg", "bg", "wo", "bo")]


class Block(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("B", "L", "C", "H", "D", "dtype")] + [
        ("eps", ctypes.c_float), ("sm_scale", ctypes.c_float), ("dropout_p", ctypes.c_float), ("seed", ctypes.c_uint64),
        ("precise", ctypes.c_int), ("z", ctypes.c_void_p), ("z_stride", ctypes.c_int64 * 3), ("mask", ctypes.c_void_p)] + _WEIGHTS


class BlockGrads(ctypes.Structure):
    _fields_ = [("z", ctypes.c_void_p), ("z_stride", ctypes.c_int64 * 3)] + _WEIGHTS


DTYPE_F16, DTYPE_BF16, DTYPE_F32 = 0, 1, 2


class FtaError(RuntimeError):
    def __init__(self, status: int, message: str):
        super().__init__(f"libfta: {message} (status {status})")
        self.status = status


_lib = None

PO = ctypes.POINTER(Options)
P5 = ctypes.POINTER(Tensor5)
P4 = ctypes.POINTER(Tensor4)
PB = ctypes.POINTER(Block)
_S3 = ctypes.POINTER(ctypes.c_int64)
_DIMS = [ctypes.c_int] * 5

SIGNATURES = {
    "fta_version": (ctypes.c_int, []),
    "fta_seq_len_supported": (ctypes.c_int, [ctypes.c_int, ctypes.c_int]),
    "fta_seq_len_supported_ex": (ctypes.c_int, [ctypes.c_int, ctypes.c_int, PO]),
    "fta_strerror": (ctypes.c_char_p, [ctypes.c_int]),
    "fta_debug_select_kernels": (ctypes.c_int, [ctypes.c_int]),
    "fta_describe_plan": (ctypes.c_int, _DIMS + [ctypes.c_char_p, ctypes.c_size_t]),
    "fta_describe_plan_ex": (ctypes.c_int, _DIMS + [ctypes.c_float, PO, ctypes.c_char_p, ctypes.c_size_t]),
    "fta_check_fwd": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p] + _DIMS + [ctypes.c_float]),
    "fta_fwd": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p] + _DIMS + [ctypes.c_float, ctypes.c_void_p]),
    "fta_bwd_workspace_bytes": (ctypes.c_size_t, _DIMS),
    "fta_bwd_workspace_bytes_ex": (ctypes.c_size_t, _DIMS + [PO]),
    "fta_fwd_ex": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p] + _DIMS + [ctypes.c_float, PO, ctypes.c_void_p]),
    "fta_bwd_ex": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p, P5, P5, P5, P5, P4, ctypes.c_void_p,
                                  ctypes.c_size_t] + _DIMS + [ctypes.c_float, PO, ctypes.c_void_p]),
    "fta_dropout_mask": (ctypes.c_int, [PO, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p,
                                        ctypes.c_void_p]),
    "fta_check_bwd": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p, P5, P5, P5, P5, P4, ctypes.c_void_p,
                                     ctypes.c_size_t] + _DIMS + [ctypes.c_float]),
    "fta_bwd": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p, P5, P5, P5, P5, P4, ctypes.c_void_p,
                               ctypes.c_size_t] + _DIMS + [ctypes.c_float, ctypes.c_void_p]),
    "fta_bwd_noalloc": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p, P5, P5, P5, P5, P4] + _DIMS
                        + [ctypes.c_float, ctypes.c_void_p]),
    "fta_bwd_profile": (ctypes.c_int, [P5, P5, P5, P4, P5, ctypes.c_void_p, P5, P5, P5, P5, P4, ctypes.c_void_p,
                                       ctypes.c_size_t] + _DIMS + [ctypes.c_float, ctypes.c_void_p,
                                                                   ctypes.POINTER(ctypes.c_float)]),
    "fta_block_check": (ctypes.c_int, [PB]),
    "fta_block_state_bytes": (ctypes.c_size_t, [PB]),
    "fta_block_bwd_workspace_bytes": (ctypes.c_size_t, [PB]),
    "fta_block_fwd": (ctypes.c_int, [PB, ctypes.c_void_p, _S3, ctypes.c_void_p, ctypes.c_void_p]),
    "fta_block_bwd": (ctypes.c_int, [PB, ctypes.c_void_p, ctypes.c_void_p, _S3, ctypes.POINTER(BlockGrads), ctypes.c_void_p,
                                     ctypes.c_size_t, ctypes.c_void_p]),
}


def load() -> ctypes.CDLL:
    """Loads the in-tree library; fails loudly when it has not been built (there is no fallback)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(
                f"{LIB_PATH} is missing: build it with `python flash-triangle-attention_amd/build.py` "
                "(hipcc, gfx950). The HIP library is the only implementation of attention().")
        lib = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _lib = lib
    return _lib


_BUILT_FOR = b"fta_native built for torch "


def native_torch_version(path: str) -> "str | None":
    """The torch version that the extension module at `path` was built for (None: no such file).  Read from the file's
    bytes: a module built for another torch must not be loaded to find out."""
    if not os.path.exists(path):
        return None
    with open(path, "rb") as f:
        data = f.read()
    a = data.find(_BUILT_FOR)
    return data[a + len(_BUILT_FOR):data.index(b"\0", a)].decode() if a >= 0 else "another build"


_native = None


def native():
    """The C++ host path (csrc/fta_torch.cpp), a Python extension module next to the library; None, with one warning,
    where it is missing or was built for another torch: the Python path beside it runs the same kernels at about
    15 us more a call, and the block as separate layers."""
    global _native
    if _native is None:
        import torch
        load()
        have, _native = native_torch_version(NATIVE_PATH), False
        try:
            if have != torch.__version__:
                raise ImportError("missing" if have is None else f"built for torch {have}, this is {torch.__version__}")
            spec = importlib.util.spec_from_file_location("fta_native", NATIVE_PATH)
            mod = importlib.util.module_from_spec(spec)
            spec.loader.exec_module(mod)
            _native = mod
        except ImportError as e:
            warnings.warn(f"{NATIVE_PATH}: {e}; calls take the slower Python path. Build it with "
                          "`python flash-triangle-attention_amd/build.py`", RuntimeWarning, stacklevel=2)
    return _native or None


def strerror(status: int) -> str:
    return load().fta_strerror(int(status)).decode()


def describe_plan(B: int, H: int, L1: int, L2: int, D: int, sm_scale: float = 1.0, options: "Options | None" = None) -> dict:
    """Kernel instance, launch count, grid, block and LDS bytes per stage, and the workspace parts, for a
    call with these sizes, softmax scale and options (None: fp16, no dropout).  "fwd" has scattered_grid, scattered_block and scattered_lds
    where keys that are not neighbours in memory run other workgroups."""
    buf = ctypes.create_string_buffer(1024)
    check(load().fta_describe_plan_ex(B, H, L1, L2, D, float(sm_scale), ctypes.byref(options) if options is not None else None,
                                      buf, len(buf)))
    out = {}
    for line in buf.value.decode().strip().split("\n"):
        stage, rest = line.split(": ", 1)
        fields = rest.split(" ")
        d = {"kernel": fields[0]} if "=" not in fields[0] else {}
        d.update({k: (int(v) if v.lstrip("-").isdigit() else v) for k, v in (f.split("=") for f in fields if "=" in f)})
        out[stage] = d
    return out


def check(status: int) -> None:
    if status != 0:
        raise FtaError(status, strerror(status))


def t5(ptr: int, strides) -> Tensor5:
    return Tensor5(ptr, (ctypes.c_int64 * 4)(*[int(s) for s in strides[:4]]))


def t4(ptr: int, strides) -> Tensor4:
    return Tensor4(ptr, (ctypes.c_int64 * 3)(*[int(s) for s in strides[:3]]))
