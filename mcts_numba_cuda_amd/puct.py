"""Host side of the PUCT select / backup path: a ctypes binding of libpuct_hip.so (C ABI: include/puct_select.h) with
the calling convention of the reference's binding, src/puct/puct_gpu_v3_cpp.py:118-156 — `launch_select(d, ...)` takes
a dictionary of device arrays — here hipmem.DeviceArray objects or torch tensors on the GPU instead of numba device
arrays.  There is no CPU fallback: without the library, or with arrays that are not on the GPU, every call raises.

When torch is used in the same process, import torch before this package: torch ships its own copy of the HIP
runtime, and the copy that is loaded first serves both."""
import ctypes
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libpuct_hip.so")

# packing of the selection word, src/puct/puct_gpu_v3.py:14-48
NODE_EXPANDED_TERMINAL = -1
PACKED_NODE_LIMIT = 16384
PACKED_NODE_MASK = 0x3FFF
PACKED_EDGE_MASK = 0xFF
PACKED_SLOT_SHIFT = 14
PACKED_KIND_SHIFT = 22
PACKED_KIND_MASK = 0x7
PACKED_REASON_SHIFT = 25
SELECT_INVALID, SELECT_EXPAND, SELECT_TERMINAL, SELECT_DEPTH_LIMIT, SELECT_BUSY = range(5)
PACKED_INVALID = (SELECT_INVALID << PACKED_KIND_SHIFT) | PACKED_NODE_MASK
REASON_UNSET, REASON_OK_EXPAND, REASON_OK_TERMINAL, REASON_OK_DEPTH_LIMIT = 0, 1, 2, 3
REASON_BUSY_EXPAND_INFLIGHT, REASON_BUSY_WINNER_RECALC = 4, 5
REASON_INVALID_SHAPE, REASON_INVALID_NODE_INFO, REASON_INVALID_NO_VALID_EDGE = 10, 11, 14
REASON_INVALID_CHILD_OOB, REASON_INVALID_UNKNOWN = 15, 16

_LIB = None


def _lib():
    global _LIB
    if _LIB is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(f"{LIB_PATH} is missing: build it with `python -m mcts_numba_cuda_amd.build` "
                               "(there is no CPU fallback for PUCT select/backup)")
        lib = ctypes.CDLL(LIB_PATH)
        c_void, c_int, c_float = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
        lib.puct_select_winner_recalc_launch.argtypes = [c_float] * 3 + [c_int] + [c_void] * 11 + [c_int] * 5 + [c_void]
        lib.puct_select_winner_recalc_launch.restype = c_int
        lib.puct_cpp_cuda_error_string.argtypes = [c_int]
        lib.puct_cpp_cuda_error_string.restype = ctypes.c_char_p
        lib.puct_edge_backup_launch.argtypes = [c_int] + [c_void] * 9 + [c_int] * 5 + [c_void]
        lib.puct_edge_backup_launch.restype = c_int
        for fn in (lib.puct_node_select_preclaim_launch, lib.puct_node_select_winner_recalc_launch):
            fn.argtypes = [c_float] * 3 + [c_void] * 11 + [c_int] * 5 + [c_void]
            fn.restype = c_int
        lib.puct_node_backup_launch.argtypes = [c_int] + [c_void] * 10 + [c_int] * 5 + [c_void]
        lib.puct_node_backup_launch.restype = c_int
        _LIB = lib
    return _LIB


def is_available():
    try:
        _lib()
        return True
    except (OSError, RuntimeError):
        return False


def decode(raw):
    """(kind, slot, node) of a packed selection word (src/puct/test_puct_gpu_v3.py:78-82)."""
    raw = int(raw)
    return ((raw >> PACKED_KIND_SHIFT) & PACKED_KIND_MASK, (raw >> PACKED_SLOT_SHIFT) & PACKED_EDGE_MASK,
            raw & PACKED_NODE_MASK)


def reason(raw):
    return (int(raw) >> PACKED_REASON_SHIFT) & 0x3F


# The arrays of a call: name -> (element type, shape).  A selection and its backup take a dozen microseconds on a GPU when
# they are small, and a call used to spend twenty on looking its arrays over: one pass over them now, each attribute asked
# once, and plain integers for ctypes.  The usual case, torch tensors that fit, goes through _puct_call (csrc/puct_call.c)
# where it has been built, which makes the same checks in C.
_TREES, _NODES, _EDGES, _WALKS, _PATHS = range(5)      # [trees], [trees, nodes], [.., edges], [trees, warps], [.., path_depth]
_ARRAYS = {"edge_child": (np.int32, _EDGES), "edge_prior": (np.float32, _EDGES), "edge_w": (np.float32, _EDGES), "edge_n": (np.int32, _EDGES),
           "edge_inflight": (np.int32, _EDGES), "node_inflight": (np.int32, _NODES), "node_expand_inflight": (np.int32, _NODES),
           "node_expanded": (np.int32, _NODES), "node_count": (np.int32, _TREES), "out_selected": (np.int32, _WALKS),
           "out_path": (np.int32, _PATHS), "out_len": (np.int32, _WALKS), "path_edge_values": (np.float32, _PATHS)}
_SHAPE_TEXT = {_TREES: "[trees]", _NODES: "[trees, nodes]", _EDGES: "[trees, nodes, edges]", _WALKS: "[trees, warps]", _PATHS: "[trees, warps, path_depth]"}


def _fields(what, *names):
    """(fields in the order of a launcher's arguments, other arrays whose shape is checked if the dictionary has them, and
    both with the launcher's number as _puct_call takes them)"""
    checked = ("edge_prior", "edge_w", "edge_n", "edge_inflight", "node_expand_inflight", "node_expanded", "node_inflight", "node_count",
               "out_selected", "out_len")
    others = tuple(n for n in checked if n not in names)
    return (tuple((n, *_ARRAYS[n]) for n in names), tuple((n, _ARRAYS[n][1]) for n in others), what,
            tuple((n, int(_ARRAYS[n][0] is np.float32), _ARRAYS[n][1]) for n in names + others))


_SELECT = _fields(0, "edge_child", "edge_prior", "edge_w", "edge_n", "edge_inflight", "node_expand_inflight", "node_expanded", "node_count",
                  "out_selected", "out_path", "out_len")
_NODE_SELECT = _fields(1, "edge_child", "edge_prior", "edge_w", "edge_n", "node_inflight", "node_expand_inflight", "node_expanded", "node_count",
                       "out_selected", "out_path", "out_len")
_EDGE_BACKUP = _fields(2, "edge_w", "edge_n", "edge_inflight", "node_expand_inflight", "node_count", "out_selected", "out_path", "out_len")
_NODE_BACKUP = _fields(3, "edge_child", "edge_w", "edge_n", "node_inflight", "node_expand_inflight", "node_count", "out_selected", "out_path", "out_len")
_torch = None                 # the torch module, once a torch tensor has been seen
_TORCH_TYPES = {}
try:
    from . import _puct_call
except ImportError:           # (host code only: without it the launchers below do the same in Python)
    _puct_call = None
_ENTRIES = {}                 # launcher -> address
_raw_stream = None            # handle of a device's current stream, without a Stream object around it where torch offers that


def _bind_torch():
    global _torch, _raw_stream
    if _torch is None:
        import torch
        _raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (lambda device: torch.cuda.current_stream(device).cuda_stream)
        _TORCH_TYPES.update({np.int32: torch.int32, np.float32: torch.float32})
        if _puct_call is not None:
            _puct_call.setup(torch.Tensor, torch.int32, torch.float32, getattr(torch._C, "_cuda_getDevice", None) or torch.cuda.current_device, _raw_stream)
        _torch = torch
    return _torch


def _device_ptr(t, dtype, name):
    """Device address of a contiguous array of `dtype`: a hipmem.DeviceArray or a torch tensor on the GPU."""
    from .hipmem import DeviceArray
    if isinstance(t, DeviceArray):
        if t.dtype != np.dtype(dtype):
            raise ValueError(f"{name}: expected {np.dtype(dtype)}, got {t.dtype}")
        return t.data_ptr()
    torch = _bind_torch()
    want = _TORCH_TYPES[dtype]
    if not isinstance(t, torch.Tensor) or not t.is_cuda or t.dtype != want or not t.is_contiguous():
        raise ValueError(f"{name}: expected a contiguous {want} tensor on the GPU")
    return t.data_ptr()


def _shape_error(name, kind):
    if name in ("out_selected", "out_len"):
        return ValueError("out_selected / out_len must have shape [trees, warps]")
    return ValueError(f"{name} must have shape {_SHAPE_TEXT[kind]}")


def _arguments(d, fields, values=None):
    """(addresses of the arrays of `fields`, (trees, nodes, edges, warps, path_depth, stream)): everything a launcher takes
    from the dictionary, checked.  `values`: path_edge_values, or None."""
    trees, nodes, edges = d["edge_child"].shape
    warps, path_depth = d["out_path"].shape[1], d["out_path"].shape[2]
    shapes = ((trees,), (trees, nodes), (trees, nodes, edges), (trees, warps), (trees, warps, path_depth))
    fields, others = fields[:2]
    for name, kind in others:
        if name in d and tuple(d[name].shape) != shapes[kind]:
            raise _shape_error(name, kind)
    out = []
    tensor = _torch.Tensor if _torch is not None else None
    for name, dtype, kind in fields:
        t = d[name]
        if t.__class__ is tensor:
            if t.shape != shapes[kind] and name != "edge_child" and name != "out_path":
                raise _shape_error(name, kind)
            if t.dtype is not _TORCH_TYPES[dtype] or not t.is_cuda or not t.is_contiguous():
                _device_ptr(t, dtype, name)      # (says what is wrong)
            out.append(t.data_ptr())
        else:
            if tuple(t.shape) != shapes[kind] and name != "edge_child" and name != "out_path":
                raise _shape_error(name, kind)
            out.append(_device_ptr(t, dtype, name))
            tensor = _torch.Tensor if _torch is not None else None
    if values is not None:
        if tuple(values.shape) != shapes[_PATHS]:
            raise ValueError("path_edge_values must have shape [trees, warps, path_depth]")
        values = _device_ptr(values, np.float32, "path_edge_values")
    return out, values, trees, nodes, edges, warps, path_depth, _stream_handle(d)


def _stream_handle(d):
    """torch's current stream when the arrays are torch tensors, the default stream otherwise."""
    if _torch is not None and isinstance(d["edge_child"], _torch.Tensor):
        return _raw_stream(_torch.cuda.current_device())
    return 0


def _check(code, what):
    if code != 0:
        msg = _lib().puct_cpp_cuda_error_string(code).decode("utf-8", "replace")
        raise RuntimeError(f"PUCT {what} launch failed: {msg} ({code})")


def _launch(name, fields, d, values, whole, floats=(0.0, 0.0, 0.0)):
    """Calls the launcher `name` with the arrays of d: `whole` is its soft_winner or virtual_loss, floats its cpuct, c_pw, alpha_pw."""
    lib = _LIB or _lib()
    code = None
    if _torch is not None and _puct_call is not None:
        entry = _ENTRIES.get(name)
        if entry is None:
            entry = _ENTRIES[name] = ctypes.cast(getattr(lib, name), ctypes.c_void_p).value
        code = _puct_call.launch(fields[2], entry, fields[3], d, values, whole, *floats)
    if code is None:
        arrays, values, *rest = _arguments(d, fields, values)
        args = {0: (*floats, whole, *arrays), 1: (*floats, *arrays)}.get(fields[2]) or (whole, *arrays, values)
        code = getattr(lib, name)(*args, *rest)
    if code:
        _check(code, "edge backup" if name == "puct_edge_backup_launch" else "node backup" if name == "puct_node_backup_launch" else
               "select" if name == "puct_select_winner_recalc_launch" else "node select")


def launch_select(d, cpuct=1.0, c_pw=1.0, alpha_pw=0.5, soft_winner=0):
    """Asynchronous PUCT selection on torch's current stream (src/puct/puct_gpu_v3_cpp.py:118-156)."""
    _launch("puct_select_winner_recalc_launch", _SELECT, d, None, int(soft_winner), (cpuct, c_pw, alpha_pw))


VARIANT_PRECLAIM, VARIANT_WINNER_RECALC = "preclaim", "winner_recalc"   # src/puct/test_puct_gpu_v2.py:317-352
_NODE_SELECTS = {VARIANT_PRECLAIM: "puct_node_select_preclaim_launch", VARIANT_WINNER_RECALC: "puct_node_select_winner_recalc_launch"}


def launch_node_select(d, cpuct=1.0, c_pw=1.0, alpha_pw=0.5, variant=VARIANT_PRECLAIM):
    """Asynchronous PUCT selection with node-level virtual loss (d["node_inflight"], int32 [trees, nodes]): the two
    kernels of src/puct/puct_gpu_v2.py:573-840, chosen by `variant` as in the reference's launch helper
    (src/puct/test_puct_gpu_v2.py:317-352).  Selection words have the v2 layout (no reason field, no BUSY kind)."""
    name = _NODE_SELECTS.get(variant)
    if name is None:
        raise ValueError(f"unknown select variant: {variant}")
    _launch(name, _NODE_SELECT, d, None, 0, (cpuct, c_pw, alpha_pw))


def launch_edge_backup(d, path_edge_values=None, virtual_loss=1):
    """Releases the edge-level claims of launch_select; with `path_edge_values` (float32 [trees, warps, path_depth],
    already in the perspective of each edge's owner) it also adds one visit and the value to every path edge."""
    _launch("puct_edge_backup_launch", _EDGE_BACKUP, d, path_edge_values, int(virtual_loss))


def launch_node_backup(d, path_edge_values, virtual_loss=1):
    """Backup with node-level virtual loss (d["node_inflight"]), src/puct/puct_gpu_v2.py:847-927."""
    if path_edge_values is None:
        raise ValueError("path_edge_values must have shape [trees, warps, path_depth]")
    _launch("puct_node_backup_launch", _NODE_BACKUP, d, path_edge_values, int(virtual_loss))
