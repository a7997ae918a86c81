"""The two routes of a PUCT launch on torch tensors -- _puct_call (csrc/puct_call.c) and the Python code that takes whatever
it leaves -- driven without torch: `Tensor` has what a launch asks of a torch tensor, over a given address."""
import contextlib
import ctypes
import types

import numpy as np

INT32, FLOAT32 = "torch.int32", "torch.float32"   # (told apart by identity, as torch's types are)
DEVICE, STREAM = 3, 0x7000


class Tensor:
    def __init__(self, shape, dtype, address, is_cuda=True, contiguous=True):
        self.shape, self.dtype, self.is_cuda = tuple(shape), dtype, is_cuda
        self._address, self._contiguous = address, contiguous

    def is_contiguous(self):
        return self._contiguous

    def data_ptr(self):
        return self._address


def torch_type(dtype):
    return {np.dtype(np.int32): INT32, np.dtype(np.float32): FLOAT32}.get(np.dtype(dtype), "torch.other")


class DLTensor(ctypes.Structure):   # (as DLPack publishes it)
    _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int32), ("device_id", ctypes.c_int32), ("ndim", ctypes.c_int32),
                ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16), ("shape", ctypes.POINTER(ctypes.c_int64)),
                ("strides", ctypes.POINTER(ctypes.c_int64)), ("byte_offset", ctypes.c_uint64)]


FROM_OBJECT = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.py_object, ctypes.POINTER(DLTensor))


class ExchangeTable(ctypes.Structure):
    _fields_ = [("major", ctypes.c_uint32), ("minor", ctypes.c_uint32), ("older", ctypes.c_void_p), ("allocator", ctypes.c_void_p), ("managed_from", ctypes.c_void_p),
                ("managed_to", ctypes.c_void_p), ("tensor_from", FROM_OBJECT), ("work_stream", ctypes.c_void_p)]


def exchange_table(answers):
    """A table of one function, which describes a Tensor, as a capsule; `answers` counts the Tensors described, and keeps what has to stay."""
    def describe(t, out):
        n = len(t.shape)
        strides, step = [0] * n, 1
        for i in range(n - 1, -1, -1):
            strides[i], step = (step if t.is_contiguous() else 2 * step), step * t.shape[i]
        shape, strides = (ctypes.c_int64 * n)(*t.shape), (ctypes.c_int64 * n)(*strides)
        answers.append((shape, strides))
        o = out[0]
        # (half the address as an offset: DLPack leaves it to the framework where an array starts)
        o.data, o.byte_offset, o.ndim, o.lanes, o.bits = t.data_ptr() - t.data_ptr() // 2, t.data_ptr() // 2, n, 1, 32 if t.dtype in (INT32, FLOAT32) else 64
        o.device_type, o.device_id, o.code = 10 if t.is_cuda else 1, 0, 2 if t.dtype is FLOAT32 else 0
        o.shape, o.strides = ctypes.cast(shape, ctypes.POINTER(ctypes.c_int64)), ctypes.cast(strides, ctypes.POINTER(ctypes.c_int64))
        return 0
    table = ExchangeTable(major=1, tensor_from=FROM_OBJECT(describe))
    new = ctypes.pythonapi.PyCapsule_New
    new.restype, new.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
    name = b"dlpack_exchange_api"
    answers.append((table, name))
    return new(ctypes.addressof(table), name, None)


@contextlib.contextmanager
def routes(stream=STREAM, described=None):
    """Makes `Tensor` the tensor type of mcts_numba_cuda_amd.puct while it lasts; yields the module's _puct_call (None if not built).
    described: a list, for a Tensor type with an exchange table that notes in it what it described."""
    if described is not None:
        Tensor.__dlpack_c_exchange_api__ = exchange_table(described)
    from mcts_numba_cuda_amd import puct
    kept = puct._torch, dict(puct._TORCH_TYPES), puct._raw_stream, puct._puct_call
    current = lambda device: stream if device == DEVICE else -1
    puct._torch = types.SimpleNamespace(Tensor=Tensor, cuda=types.SimpleNamespace(current_device=lambda: DEVICE))
    puct._TORCH_TYPES.clear()
    puct._TORCH_TYPES.update({np.int32: INT32, np.float32: FLOAT32})
    puct._raw_stream = current
    if puct._puct_call is not None:
        puct._puct_call.setup(Tensor, INT32, FLOAT32, lambda: DEVICE, current)
    try:
        yield puct._puct_call
    finally:
        if described is not None:
            del Tensor.__dlpack_c_exchange_api__
            if kept[3] is not None:
                kept[3].setup(Tensor, INT32, FLOAT32, lambda: DEVICE, current)   # (lets go of the table)
        puct._torch, types_before, puct._raw_stream, puct._puct_call = kept
        puct._TORCH_TYPES.clear()
        puct._TORCH_TYPES.update(types_before)
        if kept[0] is not None:   # (torch was bound before: bind it again)
            puct._torch = None
            puct._bind_torch()
