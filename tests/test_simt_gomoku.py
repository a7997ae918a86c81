"""The Gomoku search kernels on the CPU (tests/simt: lanes that meet where the device's do, wavefronts in any order between
barriers), against the oracle."""
import ctypes
import functools
import os
import re
import struct
import subprocess

import numpy as np
import pytest

import simt_build
from helpers import random_gomoku_root
from mcts_numba_cuda_amd import _lib
from mcts_numba_cuda_amd.build import LIB
from oracle.oracle import Oracle

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
needs_clang = pytest.mark.skipif(simt_build.CLANG is None, reason="no clang++")


@functools.lru_cache(None)
def library(path):
    lib = ctypes.CDLL(path)
    lib.simt_gomoku.argtypes = [ctypes.c_int] * 11 + [ctypes.c_float, ctypes.c_int, ctypes.c_int, ctypes.c_uint, ctypes.c_void_p, ctypes.c_int] + [ctypes.c_void_p] * 6
    return lib


def words_of(m, n):
    if m <= 16 and n <= 16 and m * n <= 240:
        return 8
    return 12 if m * n <= 384 else 16


def compare(path, m, n, stones, variant, trees, playouts, steps, groups=3, per_cu=True, launches=1, prep=48, xccs=1, seed=7, room=None):
    acp, thrifty, W, A = variant.startswith("acp"), variant.endswith("thrifty"), words_of(m, n), m * n
    S = room or 1 + A * steps * launches
    o = Oracle("gomoku", (m, n), 0, A, trees, playouts, variant, ucb_c=2.0, seed=seed, max_tree_size_override=S, threads=1)
    board, turn = random_gomoku_root(np.random.default_rng(seed), m, n, stones)
    rng = o.rng_states("playout").copy()
    # (the expansion generators are those of the same seed's stream that start a tree's threads)
    tpb = 1
    while tpb < max(m * n, A):
        tpb *= 2
    tpb = min(tpb, 512)
    streams = Oracle("gomoku", (m, n), 0, A, trees * 8, 64, "acp_prodigal", seed=seed, max_tree_size_override=1).rng_states("playout")
    expand = np.ascontiguousarray(streams[np.arange(trees) * tpb])
    bits = np.zeros((2, 32 * W), np.uint8)
    bits[0, :A], bits[1, :A] = board.ravel() == 1, board.ravel() == -1
    bb = np.packbits(bits, axis=1, bitorder="little").view(np.uint32)
    rec = 256 if W > 12 else 128
    nodes, stats = np.zeros((trees, S, rec), np.uint8), np.zeros((trees, S, 4), np.int32)
    sizes, layout = np.zeros(trees, np.int32), np.zeros(3, np.int32)
    rc = library(path).simt_gomoku(m, n, trees, playouts, acp, thrifty, groups, per_cu, S, steps, launches, 2.0, prep, xccs, seed, bb.ctypes.data, turn,
                                        rng.ctypes.data, expand.ctypes.data, nodes.ctypes.data, stats.ctypes.data, sizes.ctypes.data, layout.ctypes.data)
    assert rc == 0
    o.run(board, None, turn, steps * launches)
    for t in range(trees):
        sz = o.tree_size(t)
        assert sizes[t] == sz, (t, sizes[t], sz)
        np.testing.assert_array_equal(stats[t, :sz, 0], o.tree(t, "ns"), err_msg=f"ns[{t}]")
        np.testing.assert_array_equal(stats[t, :sz, 1], o.tree(t, "ns_wins"), err_msg=f"wins[{t}]")
        head = nodes[t, :sz].view(np.int32)
        np.testing.assert_array_equal(head[:, 1], o.tree(t, "trees")[:, 0], err_msg=f"parents[{t}]")
        np.testing.assert_array_equal(nodes[t, :sz, 16:18].copy().view(np.int16)[:, 0], o.tree(t, "depths"))
        np.testing.assert_array_equal(nodes[t, 1:sz, 19].view(np.int8), o.tree(t, "outcomes")[1:])
    np.testing.assert_array_equal(rng, o.rng_states("playout"), err_msg="generators")
    return layout


# rows, columns, stones, variant, trees, playouts, steps, and how the search is laid out: formats of either side of the limit on times,
# several rounds, two trees to a CU, all wavefronts on one board of times, full pools, paths beyond what is prepared, workgroups on one XCC and on several
CASES = [
    (5, 5, 0, "acp_prodigal", 2, 64, 3, dict(groups=5, xccs=8)), (5, 32, 0, "ocp_thrifty", 1, 128, 3, {}), (9, 9, 6, "acp_thrifty", 1, 64, 4, dict(xccs=3)),
    (11, 11, 0, "acp_prodigal", 2, 32, 3, dict(groups=4, xccs=8)), (13, 13, 30, "acp_prodigal", 1, 32, 3, {}), (13, 14, 0, "ocp_prodigal", 2, 256, 4, {}),
    (15, 15, 0, "ocp_thrifty", 1, 512, 3, {}), (15, 15, 0, "ocp_prodigal", 2, 128, 6, dict(per_cu=False, launches=2)), (15, 15, 90, "acp_prodigal", 2, 32, 2, {}),
    (15, 14, 130, "ocp_thrifty", 1, 64, 8, dict(prep=2)), (10, 16, 0, "acp_thrifty", 1, 64, 2, {}), (16, 15, 3, "acp_prodigal", 1, 32, 2, dict(xccs=8)),
    (16, 16, 0, "ocp_prodigal", 1, 128, 3, {}), (17, 17, 7, "acp_prodigal", 1, 16, 2, {}), (19, 19, 100, "ocp_thrifty", 1, 128, 4, dict(prep=0)),
    (22, 23, 0, "ocp_prodigal", 1, 256, 2, {}), (32, 16, 40, "acp_thrifty", 1, 8, 2, {}), (6, 7, 40, "acp_prodigal", 1, 8, 12, {}),
    (9, 9, 4, "acp_prodigal", 1, 16, 6, dict(room=90)), (8, 8, 4, "ocp_thrifty", 1, 64, 8, dict(room=100)), (7, 7, 0, "acp_thrifty", 1, 4, 3, dict(room=1)),
    (13, 13, 0, "ocp_thrifty", 1, 32, 3, {}), (16, 16, 9, "ocp_prodigal", 1, 64, 3, {}), (32, 16, 90, "ocp_thrifty", 1, 64, 2, {}),
    (16, 16, 200, "acp_thrifty", 1, 128, 3, dict(groups=5, xccs=8)), (22, 22, 440, "acp_prodigal", 1, 2, 3, {}),
    (5, 17, 0, "acp_prodigal", 1, 64, 2, {}), (17, 5, 0, "acp_thrifty", 1, 128, 2, {}),   # (rings larger than the board of times in whose place they are)
]


@needs_clang
@pytest.mark.parametrize("case", CASES, ids=str)
def test_searches_on_the_cpu_equal_the_oracle(case):
    """With one draw in 4096 rounded up to 1.0f, so that playouts are replayed all the time."""
    simt_build.run_apart(compare, simt_build.checked("gomoku_host"), *case[:-1], **case[-1])


@needs_clang
def test_every_layout_holds_what_the_kernel_puts_there():
    """For all boards and numbers of playouts that an engine takes: the lists, the boards of times and, where two wavefronts draw, the rings of
    offsets lie within the LDS that is asked for, the rings behind the boards or (all children) in the place of the one there is; and a CU
    has that much beside what the kernel declares for itself."""
    lib = ctypes.CDLL(simt_build.checked("gomoku_host")[0])
    layout_of, of_kernel, of_cu = lib.simt_gomoku_layout, lib.simt_gomoku_kernel_lds, lib.simt_gomoku_cu_lds()
    out = (ctypes.c_int64 * 7)()
    tight = set()
    for m, n in ((m, n) for m in range(5, 33) for n in range(5, 33) if m * n <= 512):
        for playouts, acp, per_cu in ((1 << k, acp, per_cu) for k in range(10) for acp in (0, 1) for per_cu in (0, 1)):
            layout_of(m, n, playouts, acp, per_cu, out)
            threads, slots, teams, lds, lists, times, rings = out
            wide = words_of(m, n) > 8
            two_draw = wide or not acp
            assert threads in (256, 512) and slots in (64, 128, 256) and (2 if two_draw else 1) * slots <= threads, (m, n, playouts, acp, per_cu)
            assert 1 <= teams <= max(1, threads // 256) and (teams == 1 or not acp), (m, n, playouts, acp, per_cu)
            needed = lists + (times + rings if not acp else max(times, rings if wide else 0))
            assert lds >= needed, (m, n, playouts, acp, per_cu, lds, needed)
            assert lds + of_kernel(words_of(m, n), acp) <= of_cu, (m, n, playouts, acp, per_cu, lds)
            if acp and wide and rings > times:
                tight.add((m, n))
    assert tight == {(5, 17), (17, 5)}


@needs_clang
@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_the_kernels_declare_no_more_lds_than_layouts_leave_them(tmp_path):
    """The built library's own figures (its code objects' notes) against kernel_lds_bytes."""
    _lib.lib()
    with open(LIB, "rb") as f:
        data = f.read()
    at = data.index(b"__CLANG_OFFLOAD_BUNDLE__")
    entries, found = at + 32, {}
    for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):   # (offset, size, length of the target's name; the name)
        offset, size, length = struct.unpack_from("<QQQ", data, entries)
        if b"gfx950" in data[entries + 24:entries + 24 + length]:
            (tmp_path / "code").write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.check_output([READELF, "--notes", str(tmp_path / "code")], text=True)
            for kernel in re.split(r"\n  - ", notes):
                name = re.search(r"\.name: +\S*search_kernel_forINS0_6GomokuELb([01])ELi(\d+)E", kernel)
                if name:
                    found[int(name[1]), int(name[2])] = int(re.search(r"\.group_segment_fixed_size: (\d+)", kernel)[1])
        entries += 24 + length
    assert sorted(found) == [(acp, words) for acp in (0, 1) for words in (8, 12, 16)]
    most = ctypes.CDLL(simt_build.checked("gomoku_host")[0]).simt_gomoku_kernel_lds
    for (acp, words), declared in found.items():
        assert 4096 < declared <= most(words, acp), (acp, words, declared, most(words, acp))


@pytest.mark.skipif(simt_build.thread_sanitizer() is None, reason="no ThreadSanitizer")
def test_wavefronts_do_not_race():
    """No two wavefronts touch the same LDS or memory, one of them writing, without a barrier or a published word in between."""
    code, output = simt_build.races("gomoku_host", "test_simt_gomoku", CASES)
    assert code == 0, output[-6000:]
