"""The lanes of a row that hold no edge (csrc/puct_row.h, compiled for the host): whatever their slots hold, their score is
finite and below every edge's."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcts_numba_cuda_amd", "csrc")
SOURCE = """
#include "puct_row.h"
float score(int edge, float q, float cp, int den, float sqrt_parent) {
    return prow_score(prow_q(edge, q), prow_cp(edge, cp), sqrt_parent, prow_den(edge, den));
}
/* How many of `count` quotients differ from the division's in any bit, with a reciprocal that is `ulps` off the rounded one. */
int quotients_that_differ(const float *num, const int *den, int count, int ulps) {
    int wrong = 0;
    for (int i = 0; i < count; ++i) {
        union { float f; int i; } r, a, b;
        r.f = 1.0f / (float)den[i];
        r.i += ulps;
        a.f = prow_quotient(num[i], (float)den[i], r.f);
        b.f = num[i] / (float)den[i];
        wrong += a.i != b.i;
    }
    return wrong;
}
"""
INT_MIN = -2**31


@pytest.fixture(scope="module")
def row(tmp_path_factory):
    at = tmp_path_factory.mktemp("puct_row")
    (at / "row.c").write_text(SOURCE)
    lib = str(at / "row.so")
    subprocess.check_call(["gcc", "-std=c99", "-O2", "-Wall", "-Werror", "-ffp-contract=off", "-shared", "-fPIC", "-I" + CSRC, "-o", lib, str(at / "row.c"), "-lm"])
    so, f = ctypes.CDLL(lib), ctypes.c_float
    so.score.argtypes, so.score.restype = [ctypes.c_int, f, f, ctypes.c_int, f], f
    return so


@pytest.mark.parametrize("den", [0, 1, -1, 2, 255, INT_MIN, 2**31 - 1])
def test_a_lane_without_an_edge_is_finite_and_last(row, den):
    """den = 0: a slot whose words read as n = -1 and no claims.  Its quotient was 0 / 0."""
    lowest_edge = row.score(1, -1e30, -1e30, 1, float(np.sqrt(np.float32(2**31))))
    for sqrt_parent in (1.0, 2.5, float(np.sqrt(np.float32(2**31)))):
        for junk in (0.0, -0.0, 1.0, float("nan"), float("inf"), -float("inf")):
            s = row.score(0, junk, junk, den, sqrt_parent)
            assert np.isfinite(s) and s == np.float32(-np.finfo(np.float32).max), (den, junk, sqrt_parent)
            assert s < lowest_edge


@pytest.mark.parametrize("ulps", [-1, 0, 1])
def test_the_short_division_is_the_division(row, ulps):
    """Every bit, over the declared range of operands (cp of prow_cp_fits times a root of up to 2^16), small and large counts."""
    rng = np.random.default_rng(5 + ulps)
    for low, high in ((1, 64), (1, 70000), (1, 2**24), (2**24, 2**31 - 64)):
        n = 400000
        num = np.exp(rng.uniform(np.log(1e-20), np.log(1e15 * 65536), n)).astype(np.float32)
        num[: n // 2] = rng.uniform(0, 300, n // 2).astype(np.float32)
        num[: n // 8] = 0.0
        den = rng.integers(low, high, n).astype(np.int32)
        p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
        assert row.quotients_that_differ(p(num), p(den), n, ulps) == 0
