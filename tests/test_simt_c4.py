"""The Connect 4 search kernels on the CPU (tests/simt), in all their forms, against the oracle."""
import ctypes
import functools

import numpy as np
import pytest

import simt_build
from helpers import random_c4_root
from oracle.oracle import Oracle

needs_clang = pytest.mark.skipif(simt_build.CLANG is None, reason="no clang++")
FORMS = ["plain", "split", "pool", "solo"]
NODE = np.dtype([("ns", "<i4", 8), ("wins", "<i4", 8), ("pos", "<u8"), ("neg", "<u8"), ("base", "<i4"), ("parent", "<i4"), ("depth", "<i2"), ("turn", "i1"),
                 ("outcome", "i1"), ("mask", "u1"), ("flags", "u1"), ("action", "u1"), ("best", "u1"), ("rest", "<u4", 8)])


@functools.lru_cache(None)
def library(path):
    lib = ctypes.CDLL(path)
    lib.simt_c4.argtypes = [ctypes.c_int] * 11 + [ctypes.c_float, ctypes.c_int, ctypes.c_int, ctypes.c_uint, ctypes.c_void_p, ctypes.c_int] + [ctypes.c_void_p] * 4
    return lib


def compare(path, m, n, plies, variant, trees, playouts, steps, form="split", threads=None, launches=1, fences=0, xccs=8, seed=7, room=None):
    acp, thrifty = variant.startswith("acp"), variant.endswith("thrifty")
    S = room or 1 + n * steps * launches
    o = Oracle("c4", (m, n), n, n, trees, playouts, variant, ucb_c=2.0, seed=seed, max_tree_size_override=S, threads=1)
    board, fills, turn = random_c4_root(np.random.default_rng(seed), plies, m, n)
    rng = o.rng_states("playout").copy()
    tpb = 1   # (the expansion generators are those of the same seed's stream that start a tree's threads)
    while tpb < max(m * n, n):
        tpb *= 2
    streams = Oracle("c4", (m, n), n, n, trees, 64, "acp_prodigal", seed=seed, max_tree_size_override=1).rng_states("playout")
    expand = np.ascontiguousarray(streams[np.arange(trees) * tpb])
    bb = np.zeros(2, np.uint64)
    for j in range(n):
        for r in range(m):
            v = board[m - 1 - r, j]
            if v:
                bb[0 if v == 1 else 1] |= np.uint64(1 << (j * (m + 1) + r))
    nodes, sizes = np.zeros((trees, S), NODE), np.zeros((trees, 3), np.int32)
    threads = threads or max(64, min(playouts, 512))
    rc = library(path).simt_c4(m, n, trees, playouts, acp, thrifty, FORMS.index(form), threads, S, steps, launches, 2.0, fences, xccs, seed, bb.ctypes.data, turn,
                                    rng.ctypes.data, expand.ctypes.data, nodes.ctypes.data, sizes.ctypes.data)
    assert rc == 0, "given up"
    o.run(board, fills, turn, steps * launches)
    for t in range(trees):
        sz = o.tree_size(t)
        assert sizes[t, 0] == sz, (t, sizes[t], sz)
        d = nodes[t, :sz]
        np.testing.assert_array_equal(d["parent"], o.tree(t, "trees")[:, 0], err_msg=f"parents[{t}]")
        for name, theirs, root in (("ns", "ns", sizes[t, 1]), ("wins", "ns_wins", sizes[t, 2])):
            mine = np.concatenate([[root], d[name][d["parent"][1:], d["action"][1:]]])
            np.testing.assert_array_equal(mine, o.tree(t, theirs), err_msg=f"{theirs}[{t}]")
        np.testing.assert_array_equal(d["depth"], o.tree(t, "depths"))
        np.testing.assert_array_equal(d["outcome"][1:], o.tree(t, "outcomes")[1:])
    np.testing.assert_array_equal(rng, o.rng_states("playout"), err_msg="generators")


CASES = [  # rows, columns, plies, variant, trees, playouts, steps, and how the search is laid out
    (6, 7, 0, "ocp_thrifty", 1, 64, 60, {}), (8, 6, 1, "ocp_prodigal", 2, 32, 30, {}), (4, 4, 9, "ocp_thrifty", 1, 1, 100, dict(launches=2)),
    (6, 7, 0, "acp_prodigal", 1, 64, 15, {}), (7, 8, 0, "acp_thrifty", 1, 256, 4, {}), (6, 7, 30, "acp_thrifty", 1, 128, 60, {}),
    (6, 7, 30, "acp_prodigal", 1, 64, 120, dict(fences=1, launches=2)), (5, 8, 22, "acp_prodigal", 1, 64, 60, dict(xccs=3)), (4, 4, 0, "acp_prodigal", 2, 64, 250, {}),
    (13, 1, 9, "acp_prodigal", 1, 128, 40, {}), (6, 7, 26, "acp_thrifty", 1, 64, 60, dict(room=50)),
    (6, 7, 0, "acp_prodigal", 2, 64, 10, dict(form="plain")), (6, 7, 26, "acp_thrifty", 1, 128, 60, dict(form="plain", fences=1)), (4, 8, 0, "acp_thrifty", 1, 32, 20, dict(form="plain", threads=128)),
    (6, 7, 0, "ocp_prodigal", 2, 128, 30, dict(form="plain", threads=256)), (6, 7, 0, "acp_prodigal", 1, 128, 10, dict(form="pool", threads=64)), (7, 7, 10, "acp_thrifty", 2, 64, 10, dict(form="solo", threads=128)),
]


@needs_clang
@pytest.mark.parametrize("case", CASES, ids=str)
def test_searches_on_the_cpu_equal_the_oracle(case):
    """With one draw in 4096 rounded up to 1.0f, so that playouts are replayed all the time."""
    simt_build.run_apart(compare, simt_build.checked("c4_host"), *case[:-1], **case[-1])


@pytest.mark.skipif(simt_build.thread_sanitizer() is None, reason="no ThreadSanitizer")
def test_wavefronts_do_not_race():
    """No two wavefronts touch the same LDS or memory, one of them writing, without a barrier or a published word in between
    (but split_choose, which reads draws ahead of those made: it uses them only for moves beyond the board's last)."""
    code, output = simt_build.races("c4_host", "test_simt_c4", [c for c in CASES if c[5] <= 128 and c[6] <= 120], "split_choose")
    assert code == 0, output[-6000:]
