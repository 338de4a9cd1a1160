"""ctypes binding of libe3x.so, the C ABI of the HIP kernels.

The library is built in-tree by ``e3nn_amd.csrc.build``; nothing here falls back to
another implementation: if the shared object is missing, importing a symbol raises.
"""
import contextlib
import ctypes
import importlib.util
import os

import torch  # loads the HIP runtime the library links against
from torch.autograd import forward_ad

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "lib", "libe3x.so")
HOST_PATH = os.path.join(_HERE, "lib", "_e3x_host.so")

F32, BF16 = 0, 1
MODE_UVW, MODE_UVU = 0, 1
NORM_INTEGRAL, NORM_COMPONENT, NORM_NORM = 0, 1, 2
ERR_INDEX = -4
ERR_INVALID = -1
ERR_COMPILE = -2

c_void_p, c_int, c_int32, c_int64, c_size_t = ctypes.c_void_p, ctypes.c_int, ctypes.c_int32, ctypes.c_int64, ctypes.c_size_t


class Irrep(ctypes.Structure):
    _fields_ = [("mul", c_int32), ("l", c_int32), ("p", c_int32)]


class Instruction(ctypes.Structure):
    _fields_ = [("i_in1", c_int32), ("i_in2", c_int32), ("i_out", c_int32), ("mode", c_int32),
                ("has_weight", c_int32), ("path_weight", ctypes.c_double)]  # fmt: skip


class TpDesc(ctypes.Structure):
    _fields_ = [("n_in1", c_int32), ("n_in2", c_int32), ("n_out", c_int32), ("n_ins", c_int32),
                ("in1", ctypes.POINTER(Irrep)), ("in2", ctypes.POINTER(Irrep)), ("out", ctypes.POINTER(Irrep)),
                ("ins", ctypes.POINTER(Instruction)), ("shared_weights", c_int32), ("dtype", c_int32)]  # fmt: skip


_SIGNATURES = {
    "e3x_last_error": (ctypes.c_char_p, []),
    "e3x_version": (c_int, []),
    "e3x_wigner_3j": (c_int, [c_int, c_int, c_int, ctypes.POINTER(ctypes.c_double)]),
    "e3x_tp_plan_create": (c_int, [ctypes.POINTER(TpDesc), ctypes.POINTER(c_void_p)]),
    "e3x_tp_plan_destroy": (c_int, [c_void_p]),
    "e3x_tp_plan_info": (c_int, [c_void_p, ctypes.POINTER(c_int64), ctypes.POINTER(c_int64), ctypes.POINTER(c_int64),
                                 ctypes.POINTER(c_int64), ctypes.POINTER(ctypes.c_char_p), ctypes.POINTER(ctypes.c_char_p)]),
    "e3x_tp_plan_arithmetic": (ctypes.c_char_p, [c_void_p, c_int]),
    "e3x_tp_forward": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p]),
    "e3x_tp_forward_workspace_bytes": (c_size_t, [c_void_p]),
    "e3x_tp_forward_workspace_bytes_for": (c_size_t, [c_void_p, c_int64]),
    "e3x_tp_forward_ws": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_size_t, c_void_p]),
    "e3x_csr_workspace_bytes": (c_size_t, [c_int64, c_int64]),
    "e3x_csr_build": (c_int, [c_void_p, c_int, c_int64, c_int64, c_void_p, c_void_p, c_void_p, c_size_t, c_void_p]),
    "e3x_csr_static_scratch_bytes": (c_size_t, []),
    "e3x_csr_build_static": (c_int, [c_void_p, c_int, c_int64, c_int64, c_void_p, c_void_p, c_void_p]),
    "e3x_edges_workspace_bytes": (c_size_t, [c_int64, c_int64]),
    "e3x_edges_build": (c_int, [c_void_p, c_int, c_void_p, c_int, c_int64, c_int64, c_int64, c_void_p, c_void_p, c_void_p,
                                ctypes.POINTER(c_int32), ctypes.POINTER(c_int32), c_void_p, c_size_t, c_void_p]),
    "e3x_index_check": (c_int, [c_void_p, c_int, c_int64, c_int64, c_void_p]),
    "e3x_tp_gather_scatter": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                      c_void_p, c_int64, c_int64, c_int64, c_void_p]),
    "e3x_row_order_workspace_bytes": (c_size_t, [c_int64]),
    "e3x_row_order_build": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_void_p,
                                    ctypes.POINTER(c_int32), c_void_p, c_size_t, c_void_p]),
    "e3x_tp_gather_scatter_ordered": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                              c_void_p, c_void_p, c_int64, c_int64, c_int64, c_void_p]),
    "e3x_tp_gather_scatter_workspace_bytes": (c_size_t, [c_void_p, c_int64]),
    "e3x_tp_gather_scatter_ws": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                         c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_void_p, c_size_t, c_void_p]),
    "e3x_tp_plan_prepare_gather_scatter_sh": (c_int, [c_void_p, c_int32, c_int32]),
    "e3x_tp_gather_scatter_sh": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                         c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int32, c_int32, c_void_p]),
    "e3x_src_rows_build": (c_int, [c_void_p, c_int, c_void_p, c_int64, c_int64, c_void_p, c_void_p]),
    "e3x_tp_gather_scatter_radial": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int32, c_int32, c_int32,
                                             ctypes.c_double, ctypes.c_double, ctypes.c_double, c_void_p, c_int, c_void_p,
                                             c_void_p, c_void_p, c_int64, c_int64, c_int64, c_void_p]),
    "e3x_tp_plan_prepare_radial": (c_int, [c_void_p, c_int32, c_int32, c_int32, ctypes.c_double, ctypes.c_double, ctypes.c_double]),
    "e3x_tp_backward_w_x2": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                                     c_void_p, c_int64, c_int64, c_int64, c_void_p]),
    "e3x_tp_plan_prepare_backward_w": (c_int, [c_void_p]),
    "e3x_tp_plan_prepare_gather_scatter_grad_w": (c_int, [c_void_p]),
    "e3x_tp_gather_scatter_grad_w": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                                             c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64,
                                             c_int64, c_void_p]),
    "e3x_tp_plan_prepare_message_backward": (c_int, [c_void_p]),
    "e3x_tp_message_backward_workspace_bytes": (c_size_t, [c_void_p, c_int64]),
    "e3x_tp_message_backward": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                        c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64,
                                        c_int64, c_void_p, c_size_t, c_void_p]),
    "e3x_tp_backward_w_uvw": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p]),
    "e3x_tp_backward_w_uvw_bf16_values": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p]),
    "e3x_tp_plan_prepare_backward_w_bf16_values": (c_int, [c_void_p]),
    "e3x_mix_forward": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_void_p]),
    "e3x_mix_backward": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_void_p]),
    "e3x_gate_forward": (c_int, [c_void_p, c_int32, c_void_p, c_int32, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int32, c_void_p]),
    "e3x_gate_backward": (c_int, [c_void_p, c_int32, c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int32, c_void_p]),
    "e3x_gate_backward2": (c_int, [c_void_p, c_int32, c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64,
                                   c_int64, c_int64, c_int32, c_void_p]),
    "e3x_sh_forward": (c_int, [ctypes.POINTER(c_int32), c_int32, c_int32, c_int32, c_void_p, c_void_p, c_int64,
                               c_int32, c_void_p]),
    "e3x_sh_backward": (c_int, [ctypes.POINTER(c_int32), c_int32, c_int32, c_int32, c_void_p, c_void_p, c_void_p, c_int64,
                                c_int32, c_void_p]),
    "e3x_sh_backward2": (c_int, [ctypes.POINTER(c_int32), c_int32, c_int32, c_int32, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                 c_int64, c_int32, c_void_p]),
    "e3x_fc_plan_create": (c_int, [ctypes.POINTER(c_int32), c_int32, c_int32, ctypes.c_double, c_int32, ctypes.c_double,
                                   ctypes.c_double, c_int32, ctypes.POINTER(c_void_p)]),
    "e3x_fc_plan_create_fused": (c_int, [ctypes.POINTER(c_int32), c_int32, c_int32, ctypes.c_double, c_int32, ctypes.c_double,
                                         ctypes.c_double, c_int32, c_int32, ctypes.c_double, c_int32, ctypes.c_double,
                                         ctypes.POINTER(c_void_p)]),
    "e3x_fc_forward_epilogue": (c_int, [c_void_p, c_void_p, ctypes.POINTER(c_void_p), c_void_p, c_void_p, c_int64, c_void_p,
                                        c_size_t, c_void_p]),
    "e3x_fc_plan_destroy": (c_int, [c_void_p]),
    "e3x_fc_workspace_bytes": (c_size_t, [c_void_p]),
    "e3x_fc_plan_key": (ctypes.c_char_p, [c_void_p]),
    "e3x_fc_forward": (c_int, [c_void_p, c_void_p, ctypes.POINTER(c_void_p), c_void_p, c_int64, c_void_p, c_size_t, c_void_p]),
    "e3x_fc_plan_prepare_backward_w": (c_int, [c_void_p]),
    "e3x_fc_backward_w": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p]),
    "e3x_copy_bytes": (c_int, [c_void_p, c_void_p, c_size_t, c_void_p]),
    "e3x_stream_rows": (c_int, [c_void_p, c_size_t, c_int64, c_void_p, c_size_t, c_void_p]),
}  # fmt: skip

_lib = None


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `python -m e3nn_amd.csrc.build` "
                "(there is no fallback implementation)"
            )
        handle = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype, fn.argtypes = res, args
        _lib = handle
    return _lib


class E3xError(RuntimeError):
    pass


_native = None
_hooks = {"E3xError": E3xError}


def connect(functions):
    """Gives the host path the Python functions that it calls, by name."""
    _hooks.update(functions)
    if _native is not None:
        _native.connect(functions)


def native():
    """The extension module of the host path (csrc/host.cpp)."""
    global _native
    if _native is None:
        lib()
        if not os.path.exists(HOST_PATH):
            raise RuntimeError(f"{HOST_PATH} is missing: build it with `python -m e3nn_amd.csrc.build`")
        spec = importlib.util.spec_from_file_location("_e3x_host", HOST_PATH)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        module.connect(_hooks)
        _native = module
    return _native


def check(rc):
    if rc != 0:
        msg = lib().e3x_last_error().decode()
        if rc == ERR_INDEX:
            raise IndexError(msg)
        raise E3xError(msg)


# What a call costs on the host before its kernel is launched: a small product or a message on one molecule takes its GPU
# time several times over in Python.  So no wrapper objects where an integer does, no device switch to the device that is
# current already, no autograd node where nothing records (see `unrecorded`), and the hot calls in native code
# (csrc/host.cpp) where they need nothing of Python.  One molecule's message 19.5 us a call, 13.1 with less Python, 8.4 native;
# a small dense layer 29.5, 12.1, 6.0; harmonics of 1.9 M vectors with gradient 127, 91, 44.
def stream_ptr(device):
    """Raw handle of the current stream of ``device``."""
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if device.index is None else device.index)


_SAME_DEVICE = contextlib.nullcontext()


def on_device(device):
    """``torch.cuda.device(device)``, a no-op when it is the current device."""
    return _SAME_DEVICE if device.index is None or device.index == torch.cuda.current_device() else torch.cuda.device(device)


def ptr(t):
    return t.data_ptr() if t is not None and t.numel() > 0 else None


def unrecorded(*tensors):
    """Whether a call on these tensors is neither recorded nor transformed by anything: no gradient wanted, no forward-mode
    level open, no function transform, no tracing.  A kernel may then be called without its autograd function."""
    if torch.is_grad_enabled():
        for t in tensors:
            if t.requires_grad:
                return False
    return forward_ad._current_level < 0 and not torch._C._are_functorch_transforms_active() and torch._C._get_tracing_state() is None
