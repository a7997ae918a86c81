"""The ordinal that a Connect 4 playout draws (csrc/c4_draw.h, compiled for the host) against the reference's arithmetic
(src/mctsnc.py:2061: float32((x >> 11) * 2^-53), then a float32 product with the number of legal columns, truncated), and the
draws that round up to 1.0f."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcts_numba_cuda_amd", "csrc")
SOURCE = """
#include "c4_draw.h"
void draws(const uint64_t *outputs, float *out, long n) { for (long i = 0; i < n; i++) out[i] = c4_draw(outputs[i]); }
"""


@pytest.fixture(scope="module")
def draws(tmp_path_factory):
    import ctypes
    at = tmp_path_factory.mktemp("c4_draw")
    (at / "draw.c").write_text(SOURCE)
    lib = str(at / "draw.so")
    subprocess.check_call(["gcc", "-std=c99", "-O2", "-Wall", "-Werror", "-ffp-contract=off", "-shared", "-fPIC", "-I" + CSRC, "-o", lib, str(at / "draw.c")])
    fn = ctypes.CDLL(lib).draws
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long]

    def call(outputs):
        out = np.empty(outputs.shape, np.float32)
        fn(outputs.ctypes.data, out.ctypes.data, outputs.size)
        return out
    return call


def around(value, reach=2000):
    """Outputs on both sides of one: single steps of its last bit, of the 53 bits that count, of a float32 near it."""
    steps = np.concatenate([np.arange(-reach, reach + 1)] + [np.arange(-reach, reach + 1) << s for s in (11, 31, 32, 36, 39)])
    near = [value + int(s) for s in steps]
    return [v for v in near if 0 <= v < 2**64]


@pytest.mark.parametrize("count", range(1, 9))
def test_ordinals_are_the_references(draws, count):
    rng = np.random.default_rng(count)
    values = [v for k in range(count + 1) for v in around((k << 64) // count)]
    values += [(1 << e) + int(d) for e in range(20, 64) for d in rng.integers(0, 1 << 20, 50)]       # every binade
    outputs = np.concatenate([np.array(values, np.uint64), rng.integers(0, 2**64, 200000, np.uint64)])
    uniform = ((outputs >> np.uint64(11)).astype(np.float64) * 2.0**-53).astype(np.float32)
    wanted = (uniform * np.float32(count)).astype(np.int64)
    draw = draws(outputs)
    rounded_up = draw >= np.float32(2**32)
    assert np.array_equal(rounded_up, uniform == 1.0) and (rounded_up.any() and not rounded_up.all())
    # what a ply computes: the draw times the count that is kept times 2^-32
    ordinal = (draw * (np.float32(count) * np.float32(2.0**-32))).astype(np.int64)
    assert np.array_equal(ordinal, wanted)
    from_2_25 = outputs >= np.uint64(1 << 57)                                                          # there the draw itself is the uniform
    assert np.array_equal(draw[from_2_25] * np.float32(2.0**-32), uniform[from_2_25])
