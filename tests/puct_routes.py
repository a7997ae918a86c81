"""The two routes of a PUCT launch on torch tensors -- _puct_call (csrc/puct_call.c) and the Python code that takes whatever
it leaves -- driven without torch: `Tensor` has what a launch asks of a torch tensor, over a given address."""
import contextlib
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


@contextlib.contextmanager
def routes(stream=STREAM):
    """Makes `Tensor` the tensor type of mcts_numba_cuda_amd.puct while it lasts; yields the module's _puct_call (None if not built)."""
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
        puct._torch, types_before, puct._raw_stream, puct._puct_call = kept
        puct._TORCH_TYPES.clear()
        puct._TORCH_TYPES.update(types_before)
        if kept[0] is not None:   # (torch was bound before: bind it again)
            puct._torch = None
            puct._bind_torch()
