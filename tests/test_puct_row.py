"""The scores of a row of 16 lanes (csrc/puct_row.h, compiled for the host).  Lanes that hold no edge: whatever their slots hold, their score is
finite and below every edge's.  The short division is the division, and decisions by the quick score are those by the score itself."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcts_numba_cuda_amd", "csrc")
SOURCE = """
#include "puct_row.h"
/* by: 0 decide_in_turn's, 1 row_decisions', 2 quick_row_decisions' */
float score(int by, int edge, float q, float cp, int den, float sqrt_parent) {
    const int d = prow_den(edge, den);
    const float reciprocal = 1.0f / (float)d, c = prow_cp(edge, cp);
    if (by == 0) return prow_score(prow_q(edge, q), c, sqrt_parent, d);
    if (by == 1) return prow_row_score(prow_q(edge, q), c, sqrt_parent, d, reciprocal);
    return prow_quick_score(prow_q(edge, q), c * reciprocal, sqrt_parent);
}
int fits(float cp) { return prow_cp_fits(cp); }

static unsigned state;
static int random_ulps(void) { state = state * 1664525u + 1013904223u; return (int)(state >> 16) % 3 - 1; }
static float near_reciprocal(int den) {   /* right to an ulp */
    union { float f; int i; } r;
    r.f = 1.0f / (float)den;
    r.i += random_ulps();
    return r.f;
}
/* Rows of `edges` edges, each decided `members` times running, by the quick score as quick_row_decisions does and by the score.  Returns how many
 * rows the quick way finds clear and decides otherwise; *clear: how many it finds clear; *tied: how many of them have two largest scores. */
int rows_decided_otherwise(const float *q, const float *cp, const int *den, const int *total, int rows, int edges, int members, unsigned seed, int *clear, int *tied) {
    int wrong = 0;
    state = seed;
    *clear = *tied = 0;
    for (int r = 0; r < rows; ++r, q += edges, cp += edges, den += edges) {
        float root[17], by[16], lifted[16], largest = 0.0f, lift = 0.0f;
        int d[16], taken[16], is_clear = 1;
        for (int n = 0; n <= members; ++n) root[n] = sqrtf((float)(total[r] + n > 1 ? total[r] + n : 1));
        for (int e = 0; e < edges; ++e) {
            d[e] = den[e];
            by[e] = cp[e] * near_reciprocal(d[e]);
            largest = fmaxf(largest, prow_quick_size(q[e], by[e], root[members]));
            if (q[e] < 0.0f) lift = fmaxf(lift, -q[e]);
        }
        const float apart = prow_quick_apart(largest);
        for (int e = 0; e < edges; ++e) lifted[e] = q[e] + lift;
        for (int n = 0; n < members; ++n) {
            float score[16], top = 0.0f;
            int takers = 0;
            for (int e = 0; e < edges; ++e) {
                score[e] = prow_quick_score(lifted[e], by[e], root[n]);
                top = fmaxf(top, score[e]);
            }
            for (int e = 0; e < edges; ++e)
                if (score[e] + apart >= top) {
                    takers += 1;
                    taken[n] = e;
                    d[e] += 1;
                    by[e] = cp[e] * near_reciprocal(d[e]);
                }
            is_clear &= takers == 1;
        }
        if (!is_clear) continue;
        *clear += 1;
        int bad = 0, equal = 0;
        for (int e = 0; e < edges; ++e) d[e] = den[e];
        for (int n = 0; n < members; ++n) {
            int best = 0;
            float top = prow_score(q[0], cp[0], root[n], d[0]);
            for (int e = 1; e < edges; ++e) {
                const float s = prow_score(q[e], cp[e], root[n], d[e]);
                if (s == top) equal = 1;
                if (s > top) top = s, best = e, equal = 0;
            }
            bad |= best != taken[n] || equal;
            d[best] += 1;
        }
        wrong += bad;
        *tied += equal;
    }
    return wrong;
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
    so.score.argtypes, so.score.restype = [ctypes.c_int, ctypes.c_int, f, f, ctypes.c_int, f], f
    so.fits.argtypes = [f]
    return so


@pytest.mark.parametrize("by", [0, 1, 2])
@pytest.mark.parametrize("den", [0, 1, -1, 2, 255, INT_MIN, 2**31 - 1])
def test_a_lane_without_an_edge_is_finite_and_last(row, den, by):
    """By each of the three scores.  den = 0: a slot whose words read as n = -1 and no claims.  Its quotient was 0 / 0."""
    largest_root = float(np.sqrt(np.float32(2**31)))
    lowest_edge = min(row.score(by, 1, -1e30, -1e30 if by == 0 else 0.0, 1, largest_root), 0.0 if by == 2 else 1.0)   # (a quick score is not negative)
    for sqrt_parent in (1.0, 2.5, largest_root):
        for junk in (0.0, -0.0, 1.0, float("nan"), float("inf"), -float("inf")):
            s = row.score(by, 0, junk, junk, den, sqrt_parent)
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


@pytest.mark.parametrize("ulps", [-1, 0, 1])
def test_the_short_division_at_the_ends_of_its_range(row, ulps):
    """The largest and smallest cp that fit, with the roots of 1 and of 2^31, and what is just beyond them does not fit."""
    low, high = np.float32(1e-20), np.float32(1e15)
    assert [row.fits(x) for x in (0.0, low, high, np.nextafter(high, np.float32(0)), np.float32(1.0))] == [1] * 5
    assert [row.fits(x) for x in (np.nextafter(low, np.float32(0)), np.nextafter(high, np.float32(np.inf)), -low, -1.0, float("nan"), float("inf"), np.float32(1e-45))] == [0] * 7
    den = np.array([1, 2, 3, 7, 255, 65537, 2**24 - 1, 2**24, 2**24 + 1, 2**30, 2**31 - 1], np.int32)
    for cp in (low, np.float32(1.1e-20), high, np.float32(9.9e14)):
        for root in (np.float32(1), np.sqrt(np.float32(2)), np.sqrt(np.float32(3)), np.sqrt(np.float32(2**31))):
            num = np.full(den.size, cp * root, np.float32)
            assert row.quotients_that_differ(num.ctypes.data_as(ctypes.c_void_p), den.ctypes.data_as(ctypes.c_void_p), den.size, ulps) == 0


@pytest.mark.parametrize("edges,members", [(2, 16), (3, 5), (4, 16), (5, 4), (16, 16)])
@pytest.mark.parametrize("kind", ["ordinary", "near", "apart", "negative", "tiny"])
def test_quick_decisions_are_those_by_the_score(row, edges, members, kind):
    """Wherever exactly one edge is taken by every quick decision, the scores take the same, with reciprocals an ulp off either way: ordinary rows, rows whose edges
    are nearly tied (and never quite, or they would not be clear), and terms far apart in size."""
    rng = np.random.default_rng(edges * 100 + members)
    rows = 20000
    shape = (rows, edges)
    den = rng.integers(1, 60, shape).astype(np.int32)
    cp = rng.uniform(0.001, 1.5, shape).astype(np.float32)
    q = rng.uniform(-1, 1, shape).astype(np.float32)
    total = (den.sum(1) - edges + rng.integers(0, 100, rows)).astype(np.int32)
    if kind == "near":   # scores of the first decision within some 2^-23 to 2^-15 of each other
        root = np.sqrt(np.maximum(total, 1).astype(np.float64))[:, None]
        aim = rng.uniform(0.2, 2.0, (rows, 1)) * (1 + np.exp2(rng.uniform(-23, -15, shape)) * rng.choice([-1, 1], shape))
        q = (aim - cp.astype(np.float64) * root / den).astype(np.float32)
    elif kind == "apart":
        cp = np.exp(rng.uniform(np.log(1e-20), np.log(1e15), shape)).astype(np.float32)
        cp[rng.random(shape) < 0.2] = 0.0
        q = (rng.choice([-1, 1], shape) * np.exp(rng.uniform(np.log(1e-30), np.log(1e15), shape))).astype(np.float32)
    elif kind == "negative":
        q = -rng.uniform(0.9, 1.0, shape).astype(np.float32)
        cp = (cp * 1e-3).astype(np.float32)
    elif kind == "tiny":
        cp = np.exp(rng.uniform(np.log(1e-20), np.log(1e-18), shape)).astype(np.float32)
        q = (rng.choice([-1, 0, 1], shape) * 1e-19).astype(np.float32)
        total = rng.integers(0, 2**31 - 64, rows).astype(np.int32)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    clear, tied = ctypes.c_int(), ctypes.c_int()
    wrong = row.rows_decided_otherwise(p(q), p(cp), p(den), p(total), rows, edges, members, 7, ctypes.byref(clear), ctypes.byref(tied))
    assert wrong == 0 and tied.value == 0
    assert clear.value > (50 if kind == "near" else 1000)   # (else the test says nothing)
