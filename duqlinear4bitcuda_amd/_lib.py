"""ctypes binding of libduq_hip.so (the C ABI declared in include/duq_hip.h).

The shared library is built in-tree by ``duqlinear4bitcuda_amd/csrc/Makefile`` (see
``duqlinear4bitcuda_amd.build``).  There is no fallback: if the library is missing,
loading raises and every op of this package fails.  The host side of its calls exists
twice: as Python code over ctypes, and in native code as ``_duq_host.so``, which is tied
to one Python and one torch.  Without that module everything runs through the former, with
the same results and kernels and more host time per call.
"""
from __future__ import annotations

import ctypes
import inspect
import os
import threading
import warnings

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libduq_hip.so")
HOST_PATH = os.path.join(_HERE, "_duq_host.so")

_c_u32 = ctypes.c_uint32
_c_i32 = ctypes.c_int32
_c_p = ctypes.c_void_p

# name -> argtypes; every function returns int status except where noted
PROTOTYPES = {
    "duq_abi_version": [],
    "duq_get_dual_quant_col_k": [],
    "duq_sym_quant_host": [_c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_sym_quant_host_qmax": [_c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_i32, _c_p, _c_p],
    "duq_sym_dual_quant_host": [_c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_asym_quant_host": [_c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_asym_dual_quant_host": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_quantize_rows_sym": [_c_p, _c_u32, _c_u32, ctypes.c_float, _c_i32, _c_p, _c_p, _c_p],
    "duq_quantize_rows_asym": [_c_p, _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_p],
    "duq_matmul_host_4bit": [_c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_batch_matmul_host_4bit": [_c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_u32, _c_p],
    "duq_asym_batch_dequant_host": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_batch_linear4bit_forward": [_c_i32, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32,
                                     _c_u32, _c_u32, _c_p, _c_p],
    "duq_quantize_product_workspace_bytes": [_c_i32, _c_u32, _c_u32, _c_u32, _c_u32],  # returns uint64_t
    "duq_quantize_product": [_c_i32, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_u32, ctypes.c_float, _c_i32, ctypes.c_float, _c_i32,
                             _c_p, _c_p, ctypes.c_uint64, _c_p],
    "duq_sym_dequant_host": [_c_p, _c_p, _c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_sym_dual_dequant_host": [_c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_asym_dequant_host": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_asym_dual_dequant_host": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_linear4bit_forward": [_c_i32, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32,
                               _c_u32, _c_p, _c_p],
    "duq_linear4bit_room_bytes": [_c_i32, _c_u32, _c_u32, _c_u32],  # returns uint64_t
    "duq_linear4bit_room_pays": [_c_i32, _c_u32, _c_u32, _c_u32],
    "duq_linear4bit_forward_room": [_c_i32] + [_c_p] * 11 + [_c_u32, _c_u32, _c_u32, _c_p, _c_p, ctypes.c_uint64, _c_p],
    "duq_product_path_for": [_c_i32, _c_u32, _c_u32, _c_u32, _c_u32, _c_i32],
    "duq_product_long_reads_for": [_c_u32, _c_u32],  # returns uint32_t
    "duq_gemm_kernel_for": [_c_u32, _c_u32, _c_u32],
    "duq_gemm_stream_tile_for": [_c_u32, _c_u32, _c_u32],
    "duq_quant_gemm_tile_for": [_c_u32, _c_u32, _c_u32],
    "duq_quantize_linear4bit_path_for": [_c_i32, _c_u32, _c_u32, _c_u32, _c_i32],
    "duq_gemm_plan_for": [_c_i32, _c_u32, _c_u32, _c_u32, _c_p],
    "duq_gemm_bf6_plan_for": [_c_i32, _c_u32, _c_u32, _c_u32, _c_p],
    "duq_quant_gemm8_tile_for": [_c_u32, _c_u32, _c_u32],
    "duq_gemm8_kernel_for": [_c_u32, _c_u32, _c_u32, _c_i32],
    "duq_probe_read": [_c_p, ctypes.c_uint64, _c_p, _c_p],
    "duq_quantize_linear4bit_workspace_bytes": [_c_u32, _c_u32, _c_u32],  # returns uint64_t (restype set in load())
    "duq_quantize_linear4bit_forward": [_c_i32, _c_p, ctypes.c_float, _c_i32, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32,
                                        _c_u32, _c_p, _c_p, _c_p, _c_p, ctypes.c_uint64, _c_p],
    "duq_quantize_linear4bit_forward_static": [_c_i32, _c_p, ctypes.c_float, _c_i32, _c_p, _c_p, _c_p, _c_p, _c_u32,
                                               _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_u32, _c_p],
    "duq_static_scratch_init": [],
    "duq_quantize_linear8bit_workspace_bytes": [_c_u32, _c_u32],  # returns uint64_t
    "duq_quantize_linear8bit_forward": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p,
                                        ctypes.c_uint64, _c_p],
    "duq_quantize_linear4bit_forward_layer": [_c_p, _c_p, _c_u32, _c_p, _c_p, ctypes.c_uint64, _c_p],
    "duq_quantize_linear4bit_asym_workspace_bytes": [_c_i32, _c_u32, _c_u32, _c_u32],  # returns uint64_t
    "duq_quantize_linear4bit_forward_asym": [_c_i32, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32,
                                             _c_u32, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, ctypes.c_uint64, _c_p],
    "duq_quantize_rows_asym_shifted": [_c_p, _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_p, _c_p],
    "duq_linear4bit_forward_rowsum": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32,
                                      _c_p, _c_p],
    "duq_asym_rowsum_dequant_host": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_asym_dual_rowsum_dequant_host": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p,
                                          _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_linear4bit_dual_rowsum_workspace_bytes": [_c_u32, _c_u32, _c_u32],  # returns uint64_t (restype set in load())
    "duq_linear4bit_forward_dual_rowsum": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p,
                                           _c_u32, _c_u32, _c_u32, _c_p, _c_p, ctypes.c_uint64, _c_p],
    "duq_weight_shadow_bf6": [_c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_quantize_rows_sym_bf6": [_c_p, _c_u32, _c_u32, ctypes.c_float, _c_i32, _c_p, _c_p, _c_p, _c_p],
    "duq_quantize_rows_asym_bf6": [_c_p, _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p],
    "duq_activation_shadow_bf6": [_c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_linear4bit_forward_bf6": [_c_i32, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32,
                                   _c_u32, _c_u32, _c_p, _c_p],
    "duq_linear4bit_forward_dual_rowsum_bf6": [_c_p] * 14 + [_c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_weight_quant_asym": [_c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p],
    "duq_weight_quant_asym_shifted": [_c_p, _c_u32, _c_u32, _c_u32] + [_c_p] * 8,
    "duq_weight_quant_sym": [_c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_p, _c_p],
    "duq_weight_quant_asym_8bit": [_c_p, _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_p],
    "duq_asym_quant_host_8bit": [_c_p, _c_p, _c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_matmul_host_8bit": [_c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_asym_dequant_host_hprec": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_quantize_rows_asym_8bit": [_c_p, _c_u32, _c_u32, _c_p, _c_p, _c_p, _c_p],
    "duq_weight_tile_8bit": [_c_p, _c_u32, _c_u32, _c_p, _c_p],
    "duq_linear8bit_forward_tiled": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
    "duq_linear8bit_forward": [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_u32, _c_u32, _c_u32, _c_p, _c_p],
}



class FusedLayer(ctypes.Structure):
    """``duq_fused_layer`` of include/duq_hip.h."""
    _fields_ = [("mode", _c_i32), ("clip", ctypes.c_float), ("qmax", _c_i32), ("N", _c_u32), ("K", _c_u32),
                ("w", _c_p), ("w_scale_1", _c_p), ("w_zeros_1", _c_p), ("w_scale_2", _c_p), ("w_zeros_2", _c_p),
                ("w_rowsum_adj", _c_p), ("w_rowsum_adj_2", _c_p), ("bias", _c_p)]


_lib = None
_loading = threading.RLock()   # (first calls may come from several threads)


class DuqError(RuntimeError):
    """A non-zero status from the C ABI (the reference raises RuntimeError from its
    torch checks, src/export/bindings.cpp:12-17)."""


def load():
    """Load the shared library once and attach prototypes."""
    if _lib is not None:
        return _lib
    with _loading:
        return _lib if _lib is not None else _load()


def _load():
    global _lib
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            f"{LIB_PATH} is missing: build it with `python -m duqlinear4bitcuda_amd.build` "
            "(hipcc --offload-arch=gfx950); there is no CPU or PyTorch fallback")
    lib = ctypes.CDLL(LIB_PATH)
    for name, argtypes in PROTOTYPES.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = ctypes.c_int
    lib.duq_quantize_linear4bit_workspace_bytes.restype = ctypes.c_uint64
    lib.duq_linear4bit_dual_rowsum_workspace_bytes.restype = ctypes.c_uint64
    lib.duq_quantize_linear4bit_asym_workspace_bytes.restype = ctypes.c_uint64
    lib.duq_quantize_linear8bit_workspace_bytes.restype = ctypes.c_uint64
    lib.duq_quantize_product_workspace_bytes.restype = ctypes.c_uint64
    lib.duq_linear4bit_room_bytes.restype = ctypes.c_uint64
    lib.duq_product_long_reads_for.restype = ctypes.c_uint32
    lib.duq_status_string.argtypes = [ctypes.c_int]
    lib.duq_status_string.restype = ctypes.c_char_p
    _lib = lib
    return lib


_host = None   # (False: looked for, and not to be had)


def _install_calls(native):
    """The native ``__call__`` of the module classes (``install`` in ``csrc/duq_host.cpp``)."""
    from torch.nn.modules import module as m

    from . import _HIP, nn
    from .nn import _calls
    lib = load()
    native.install(tuple(_calls.classes),
                   (m._global_forward_hooks, m._global_forward_pre_hooks, m._global_backward_hooks, m._global_backward_pre_hooks),
                   (m.Module, _calls.module_call, _calls.module_call_impl), (_HIP, _HIP._own_launch), (lib, lib._FuncPtr),
                   (nn.SymQuantizer, nn.AsymQuantizer, nn.AsymQuantizer8bit))
    for cls, kind, _ in _calls.classes:
        call = cls.__dict__.get("__call__")
        if type(call) is native.ModuleCall:   # (what inspect and help show is torch's)
            call.__name__, call.__qualname__, call.__module__ = "__call__", f"{cls.__qualname__}.__call__", cls.__module__
            call.__doc__, call.__signature__ = m.Module.__call__.__doc__, inspect.signature(m.Module.__call__)


def host():
    """The native module of the host side (``csrc/duq_host.cpp``, built beside the library), imported once; None, with a
    warning the first time, where it is missing or was built for another Python or torch: the callers' Python code does
    the same."""
    if _host is None:
        with _loading:
            if _host is None:
                _load_host()
    return _host or None


def _load_host():
    global _host
    load()
    try:
        if not os.path.exists(HOST_PATH):
            raise ImportError(f"{HOST_PATH} is missing")
        from . import _duq_host
    except ImportError as e:
        _host = False
        warnings.warn(f"{e}: calls take some microseconds more of host time each; build it with "
                      "`python -m duqlinear4bitcuda_amd.build`", RuntimeWarning, stacklevel=4)
        return
    from .tools.tensor_utils import PackedQuantizedTensor
    _duq_host.setup(PackedQuantizedTensor, check)
    _install_calls(_duq_host)
    _host = _duq_host


def check(status: int, what: str):
    if status != 0:
        msg = load().duq_status_string(status).decode()
        raise DuqError(f"{what}: {msg} (status {status})")
