"""Where a Gomoku playout's draw falls (csrc/gomoku_draw.h, compiled for the host) against the reference's arithmetic
(src/mctsnc.py:1882: float32((x >> 11) * 2^-53), then a float32 product with the number of cells left, truncated)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcts_numba_cuda_amd", "csrc")
SOURCE = """
#include "gomoku_draw.h"
void places(const uint64_t *outputs, uint64_t *out, long n, uint32_t count, uint32_t most) {
    for (long i = 0; i < n; i++) out[i] = gomoku_place(outputs[i], count, most);
}
uint32_t unsure(uint32_t most) { return gomoku_unsure(most); }
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    at = tmp_path_factory.mktemp("gomoku_draw")
    (at / "draw.c").write_text(SOURCE)
    lib = str(at / "draw.so")
    subprocess.check_call(["gcc", "-std=c99", "-O2", "-Wall", "-Werror", "-shared", "-fPIC", "-I" + CSRC, "-o", lib, str(at / "draw.c")])
    lib = ctypes.CDLL(lib)
    lib.places.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long, ctypes.c_uint32, ctypes.c_uint32]
    lib.unsure.restype = ctypes.c_uint32
    return lib


@pytest.mark.parametrize("most", [1, 2, 3, 16, 100, 225, 240, 361, 512])
def test_places_that_are_sure_are_the_references(library, most):
    rng = np.random.default_rng(most)
    for count in sorted({1, most, max(1, most - 1), max(1, most - 15), (most + 1) // 2, *rng.integers(1, most + 1, 4).tolist()}):
        # on both sides of every place's first output, in steps of the last bit, of the 53 bits, of a float32 and of the upper word,
        # to beyond the distance that makes a place unsure
        firsts = np.array([((k << 64) // count) % 2**64 for k in range(count)], np.uint64)
        steps = np.concatenate([np.arange(-40, 41) << s for s in (0, 11, 31, 32, 36, 38, 39, 40)] + [rng.integers(-(1 << 45), 1 << 45, 200)])
        outputs = np.concatenate([(firsts[:, None] + steps.astype(np.int64).view(np.uint64)[None, :]).ravel(), rng.integers(0, 2**64, 20000, np.uint64),
                                  np.uint64(2**64 - 1) - rng.integers(0, 1 << 42, 2000, np.uint64)])   # (wrapping round: outputs all the same)
        uniform = ((outputs >> np.uint64(11)).astype(np.float64) * 2.0**-53).astype(np.float32)
        wanted = (uniform * np.float32(count)).astype(np.int64)
        places = np.empty(outputs.shape, np.uint64)
        library.places(outputs.ctypes.data, places.ctypes.data, outputs.size, count, most)
        sure = (places & np.uint64(0xffffffff)) >= np.uint64(library.unsure(most))
        assert np.array_equal((places >> np.uint64(32)).astype(np.int64)[sure], wanted[sure])
        assert not sure[uniform == 1.0].any() and sure[-22000:-2000].mean() > 0.99   # (rounded up: never sure; most are)
