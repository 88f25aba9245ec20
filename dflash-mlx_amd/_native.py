"""ctypes binding of libdflash_mi355.so (the C ABI declared in include/dflash_mi355.h), and the module
that issues its common launches from native code (``host``, csrc/host.cpp).

There is no software fallback: if the library has not been built, or an entry
point reports an error, the caller gets an exception.
"""
from __future__ import annotations

import ctypes
import importlib.util
import os
from typing import Optional

import torch
from torch.autograd import forward_ad

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libdflash_mi355.so")
HOST_PATH = os.path.join(_HERE, "_dflash_host.so")

ABI_VERSION = 25

BF16, FP16, FP32 = 0, 1, 2
QMM_MMA2BIG, QMM_MMA2BIG_PIPE = 0, 1
QMM_KERNEL_AUTO, QMM_KERNEL_TILE, QMM_KERNEL_STREAM, QMM_KERNEL_FASTEST = 0, 1, 2, 3
QMM_STATIC_SCRATCH_BYTES = 8 << 20  # DFLASH_QMM_STATIC_SCRATCH_BYTES
QMM_CHAIN_MAX = 16                       # DFLASH_QMM_CHAIN_MAX
QMM_ERROR_OFFSET = (16384 - 64 + 1) * 4        # DFLASH_QMM_ERROR_OFFSET
QMM_CHAIN_ERROR_OFFSET = QMM_ERROR_OFFSET      # DFLASH_QMM_CHAIN_ERROR_OFFSET
QMM_EPILOGUE_NONE, QMM_EPILOGUE_SILU_MUL = 0, 1
QMM_CHAIN_JOINT_SPLIT, QMM_CHAIN_FASTEST = 1, 4  # DFLASH_QMM_CHAIN_*
QMM_LAYOUT_ROWS, QMM_LAYOUT_PACKED = 0, 1  # DFLASH_QMM_LAYOUT_*
OPT_GDN_STEP_BY_STEP, OPT_SDPA_SPLITS, OPT_QMM_SPIN_LIMIT = 0, 1, 2  # DFLASH_OPT_*


class QmmProblem(ctypes.Structure):
    """dflash_qmm_problem of include/dflash_mi355.h."""
    _fields_ = [("x", ctypes.c_void_p), ("w_q", ctypes.c_void_p), ("scales", ctypes.c_void_p),
                ("biases", ctypes.c_void_p), ("y", ctypes.c_void_p), ("K", ctypes.c_int), ("N", ctypes.c_int),
                ("wait_for", ctypes.c_int), ("epilogue", ctypes.c_int), ("layout", ctypes.c_int)]

# every symbol include/dflash_mi355.h declares
EXPORTED_SYMBOLS = (
    "dflash_abi_version",
    "dflash_last_error",
    "dflash_set_option",
    "dflash_get_option",
    "dflash_qmm_m16_workspace_bytes",
    "dflash_qmm_m16",
    "dflash_qmm_few",
    "dflash_qmm_few_silu_mul_workspace_bytes",
    "dflash_qmm_few_silu_mul",
    "dflash_qmm_few_silu_mul_by",
    "dflash_qmm_error",
    "dflash_qmm_m16_static",
    "dflash_qmm_m16_pack_gate_up",
    "dflash_qmm_m16_chain_workspace_bytes",
    "dflash_qmm_m16_chain",
    "dflash_qmm_m16_packed_bytes",
    "dflash_qmm_m16_pack",
    "dflash_qmm_m16_packed",
    "dflash_qmm_m16_packed_by",
    "dflash_qmm_rows_workspace_bytes",
    "dflash_qmm_rows",
    "dflash_qmm_m16_gather_workspace_bytes",
    "dflash_qmm_m16_gather",
    "dflash_qmm_m16_gather_by",
    "dflash_tape_replay",
    "dflash_gdn_forward_tape",
    "dflash_gdn_forward_tape_norm",
    "dflash_gdn_forward_workspace_bytes",
    "dflash_gdn_forward",
    "dflash_gdn_prepare",
    "dflash_gdn_prepare_rows",
    "dflash_gdn_block",
    "dflash_gdn_gated_norm",
    "dflash_attn_prepare",
    "dflash_attn_gate",
    "dflash_sdpa_q16_workspace_bytes",
    "dflash_sdpa_q16",
    "dflash_sdpa_q16_gated",
    "dflash_attn_block_workspace_bytes",
    "dflash_attn_block",
    "dflash_conv_state_rebuild",
    "dflash_rollback_layer",
    "dflash_rollback_layers",
)


class NativeLibraryError(RuntimeError):
    """The HIP library is missing, mismatched, or one of its calls failed."""


_lib: Optional[ctypes.CDLL] = None


def _declare(lib: ctypes.CDLL) -> None:
    c = ctypes
    lib.dflash_abi_version.restype = c.c_int
    lib.dflash_abi_version.argtypes = []
    lib.dflash_last_error.restype = c.c_char_p
    lib.dflash_last_error.argtypes = []
    lib.dflash_set_option.restype = c.c_int
    lib.dflash_set_option.argtypes = [c.c_int, c.c_int]
    lib.dflash_get_option.restype = c.c_int
    lib.dflash_get_option.argtypes = [c.c_int]
    lib.dflash_qmm_m16_workspace_bytes.restype = c.c_size_t
    lib.dflash_qmm_m16_workspace_bytes.argtypes = [c.c_int] * 6
    lib.dflash_qmm_m16.restype = c.c_int
    lib.dflash_qmm_m16.argtypes = (
        [c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 8 + [c.c_void_p]
    )
    lib.dflash_qmm_few.restype = c.c_int
    lib.dflash_qmm_few.argtypes = [c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 7 + [c.c_void_p]
    lib.dflash_qmm_few_silu_mul_workspace_bytes.restype = c.c_size_t
    lib.dflash_qmm_few_silu_mul_workspace_bytes.argtypes = [c.c_int] * 3
    lib.dflash_qmm_few_silu_mul.restype = c.c_int
    lib.dflash_qmm_few_silu_mul.argtypes = [c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 5 + [c.c_void_p]
    lib.dflash_qmm_few_silu_mul_by.restype = c.c_int
    lib.dflash_qmm_few_silu_mul_by.argtypes = [c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 6 + [c.c_void_p]
    lib.dflash_qmm_error.restype = c.c_int
    lib.dflash_qmm_error.argtypes = [c.c_void_p, c.POINTER(c.c_uint32), c.c_void_p]
    lib.dflash_qmm_m16_static.restype = c.c_int
    lib.dflash_qmm_m16_static.argtypes = [c.c_void_p] * 5 + [c.c_int] * 8 + [c.c_void_p]
    lib.dflash_qmm_m16_chain_workspace_bytes.restype = c.c_size_t
    lib.dflash_qmm_m16_chain_workspace_bytes.argtypes = [c.POINTER(QmmProblem), c.c_int, c.c_int, c.c_int]
    lib.dflash_qmm_m16_chain.restype = c.c_int
    lib.dflash_qmm_m16_chain.argtypes = [c.POINTER(QmmProblem), c.c_int, c.c_void_p, c.c_size_t] + [c.c_int] * 5 + [c.c_void_p]
    lib.dflash_qmm_m16_packed_bytes.restype = c.c_int
    lib.dflash_qmm_m16_packed_bytes.argtypes = [c.c_int] * 3 + [c.POINTER(c.c_size_t)] * 2
    lib.dflash_qmm_m16_pack.restype = c.c_int
    lib.dflash_qmm_m16_pack.argtypes = [c.c_void_p] * 6 + [c.c_int] * 3 + [c.c_void_p]
    lib.dflash_qmm_m16_pack_gate_up.restype = c.c_int
    lib.dflash_qmm_m16_pack_gate_up.argtypes = [c.c_void_p] * 6 + [c.c_int] * 3 + [c.c_void_p]
    lib.dflash_qmm_m16_packed.restype = c.c_int
    lib.dflash_qmm_m16_packed.argtypes = [c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 5 + [c.c_void_p]
    lib.dflash_qmm_m16_packed_by.restype = c.c_int
    lib.dflash_qmm_m16_packed_by.argtypes = [c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 6 + [c.c_void_p]
    lib.dflash_qmm_rows_workspace_bytes.restype = c.c_size_t
    lib.dflash_qmm_rows_workspace_bytes.argtypes = [c.c_int] * 7
    lib.dflash_qmm_rows.restype = c.c_int
    lib.dflash_qmm_rows.argtypes = [c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 7 + [c.c_void_p]
    lib.dflash_qmm_m16_gather_workspace_bytes.restype = c.c_size_t
    lib.dflash_qmm_m16_gather_workspace_bytes.argtypes = [c.c_int] * 5
    lib.dflash_qmm_m16_gather.restype = c.c_int
    lib.dflash_qmm_m16_gather.argtypes = (
        [c.c_void_p] * 7 + [c.c_size_t] + [c.c_int] * 7 + [c.c_void_p]
    )
    lib.dflash_qmm_m16_gather_by.restype = c.c_int
    lib.dflash_qmm_m16_gather_by.argtypes = [c.c_void_p] * 7 + [c.c_size_t] + [c.c_int] * 8 + [c.c_void_p]
    lib.dflash_gdn_forward_tape.restype = c.c_int
    lib.dflash_gdn_forward_tape.argtypes = [c.c_void_p] * 10 + [c.c_int] * 11 + [c.c_void_p]
    lib.dflash_gdn_forward_tape_norm.restype = c.c_int
    lib.dflash_gdn_forward_tape_norm.argtypes = [c.c_void_p] * 12 + [c.c_int] * 12 + [c.c_float, c.c_void_p]
    lib.dflash_gdn_forward_workspace_bytes.restype = c.c_size_t
    lib.dflash_gdn_forward_workspace_bytes.argtypes = [c.c_int] * 8
    lib.dflash_gdn_forward.restype = c.c_int
    lib.dflash_gdn_forward.argtypes = [c.c_void_p] * 13 + [c.c_size_t] + [c.c_longlong] * 2 + [c.c_int] * 12 + [c.c_float, c.c_void_p]
    lib.dflash_gdn_prepare.restype = c.c_int
    lib.dflash_gdn_prepare.argtypes = [c.c_void_p] * 14 + [c.c_int] * 9 + [c.c_float, c.c_void_p]
    lib.dflash_gdn_prepare_rows.restype = c.c_int
    lib.dflash_gdn_prepare_rows.argtypes = ([c.c_void_p] * 15 + [c.POINTER(c.c_longlong)] + [c.c_int] * 9 +
                                            [c.c_float, c.c_void_p])
    lib.dflash_gdn_block.restype = c.c_int
    lib.dflash_gdn_block.argtypes = [c.c_void_p] * 2
    lib.dflash_gdn_gated_norm.restype = c.c_int
    lib.dflash_gdn_gated_norm.argtypes = [c.c_void_p] * 4 + [c.c_longlong] + [c.c_int] * 3 + [c.c_float, c.c_void_p]
    lib.dflash_attn_prepare.restype = c.c_int
    lib.dflash_attn_prepare.argtypes = ([c.c_void_p] * 8 + [c.c_int] * 7 + [c.POINTER(c.c_longlong)] + [c.c_float] * 3 +
                                        [c.c_int] * 3 + [c.c_void_p])
    lib.dflash_attn_gate.restype = c.c_int
    lib.dflash_attn_gate.argtypes = [c.c_void_p] * 3 + [c.c_int] * 4 + [c.c_longlong] * 5 + [c.c_int, c.c_void_p]
    lib.dflash_sdpa_q16_workspace_bytes.restype = c.c_size_t
    lib.dflash_sdpa_q16_workspace_bytes.argtypes = [c.c_int] * 5
    lib.dflash_sdpa_q16.restype = c.c_int
    lib.dflash_sdpa_q16.argtypes = ([c.c_void_p] * 6 + [c.c_size_t] + [c.c_int] * 5 + [c.c_longlong] * 6 +
                                    [c.c_float, c.c_int, c.c_void_p])
    lib.dflash_sdpa_q16_gated.restype = c.c_int
    lib.dflash_sdpa_q16_gated.argtypes = ([c.c_void_p] * 7 + [c.c_size_t] + [c.c_int] * 5 + [c.c_longlong] * 8 +
                                          [c.c_float, c.c_int, c.c_void_p])
    lib.dflash_attn_block_workspace_bytes.restype = c.c_size_t
    lib.dflash_attn_block_workspace_bytes.argtypes = [c.c_int] * 5
    lib.dflash_attn_block.restype = c.c_int
    lib.dflash_attn_block.argtypes = [c.c_void_p] * 2
    lib.dflash_tape_replay.restype = c.c_int
    lib.dflash_tape_replay.argtypes = (
        [c.c_void_p] * 6 + [c.c_int] + [c.c_void_p] + [c.c_int] * 12 + [c.c_void_p]
    )


    lib.dflash_conv_state_rebuild.restype = c.c_int
    lib.dflash_conv_state_rebuild.argtypes = [c.c_void_p] * 4 + [c.c_int] * 6 + [c.c_void_p]
    lib.dflash_rollback_layer.restype = c.c_int
    lib.dflash_rollback_layer.argtypes = [c.c_void_p] * 9 + [c.c_int] * 16 + [c.c_void_p]
    lib.dflash_rollback_layers.restype = c.c_int
    lib.dflash_rollback_layers.argtypes = [c.c_void_p] + [c.c_int] * 16 + [c.c_void_p]


def lib() -> ctypes.CDLL:
    """Load (once) and return the native library; raise if it is not there."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise NativeLibraryError(
            f"{LIB_PATH} not found: build it with `python dflash-mlx_amd/build_ext.py` "
            "(hipcc --offload-arch=gfx950); there is no fallback for the HIP path"
        )
    loaded = ctypes.CDLL(LIB_PATH)
    for name in EXPORTED_SYMBOLS:
        if not hasattr(loaded, name):
            raise NativeLibraryError(f"{LIB_PATH} does not export {name}")
    _declare(loaded)
    got = loaded.dflash_abi_version()
    if got != ABI_VERSION:
        raise NativeLibraryError(f"ABI version {got} != expected {ABI_VERSION}; rebuild the library")
    _lib = loaded
    return loaded


_host = None


def host():
    """The native launch path (csrc/host.cpp).  Its functions serve the ordinary form of a call and return
    None for everything else, which the Python that asked then does by itself."""
    return _host if _host is not None else _load_host()


def _load_host():
    global _host
    lib()  # (the module is linked against it)
    if not os.path.exists(HOST_PATH):
        raise NativeLibraryError(f"{HOST_PATH} not found: build it with `python dflash-mlx_amd/build_ext.py`")
    spec = importlib.util.spec_from_file_location("_dflash_host", HOST_PATH)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    module.bind(NativeLibraryError)
    _host = module
    return module


def is_built() -> bool:
    # (a look at the files costs microseconds)
    return _lib is not None or (os.path.exists(LIB_PATH) and os.path.exists(HOST_PATH))


def env(key: bytes) -> Optional[bytes]:
    """Value of an environment variable as the process holds it now (``os.environ.get`` encodes the name and
    decodes the value, 1 us a look; a launch looks at three)."""
    try:
        return os.environ._data.get(key)
    except AttributeError:  # an os.environ of another make
        value = os.environ.get(os.fsdecode(key))
        return None if value is None else os.fsencode(value)


_functorch_level, _tracing = torch._C._functorch.peek_interpreter_stack, torch._C._get_tracing_state
_dispatch_modes, _compiling = torch._C._len_torch_dispatch_stack, torch.compiler.is_compiling
_grad_enabled, _Tensor, _Parameter = torch.is_grad_enabled, torch.Tensor, torch.nn.Parameter


def plain(*tensors: torch.Tensor) -> bool:
    """Ordinary tensors that nothing is differentiating, tracing or batching: what a kernel that takes
    their addresses may stand in for array operators on.  The results of such a kernel have no graph, no tangent and
    no place in a trace, so every call that the array operators could also answer asks here first."""
    if (_compiling() or forward_ad._current_level >= 0 or _functorch_level() is not None or _tracing() is not None
            or _dispatch_modes()):
        return False
    for t in tensors:
        made = type(t)
        if made is not _Tensor and made is not _Parameter:
            return False
    if _grad_enabled():
        for t in tensors:
            if t.requires_grad:
                return False
    return True


def raw_stream(device) -> int:
    """Handle of the current stream of ``device`` (torch's Stream object costs microseconds per
    call to build; the handle is all the C ABI takes)."""
    index = device.index if device.index is not None else torch.cuda.current_device()
    try:
        return torch._C._cuda_getCurrentRawStream(index)
    except AttributeError:  # a torch without the raw accessor
        return torch.cuda.current_stream(device).cuda_stream


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = lib().dflash_last_error().decode("utf-8", "replace")
        raise NativeLibraryError(f"{what} failed (code {rc}): {msg}")
