"""PUCT select / backup through the C ABI of libpuct_hip.so on the GPU: the reference's known answers, bit-exact
agreement with the sequential oracle wherever a launch is deterministic (one traversal per tree), and the invariants
every interleaving satisfies where it is not."""
import copy

import numpy as np
import pytest

import puct_cases as pc
from oracle import puct_oracle as po

pytestmark = pytest.mark.gpu


def to_device(case):
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    return {k: DeviceArray(v) for k, v in case.items()}


def to_host(d):
    return {k: v.numpy() for k, v in d.items()}


def synchronize():
    from mcts_numba_cuda_amd.hipmem import synchronize as sync
    sync()


class HipRunner(pc.Runner):
    def select(self, case, **params):
        from mcts_numba_cuda_amd import puct
        self.d = to_device(case)
        puct.launch_select(self.d, **params)
        synchronize()
        return to_host(self.d)

    def release(self):
        return self.backup(None)

    def backup(self, values):
        from mcts_numba_cuda_amd import puct
        from mcts_numba_cuda_amd.hipmem import DeviceArray
        puct.launch_edge_backup(self.d, None if values is None else DeviceArray(values))
        synchronize()
        return to_host(self.d)


@pytest.mark.parametrize("case", pc.ALL_CASES, ids=lambda f: f.__name__)
def test_known_answers(case):
    case(HipRunner())


@pytest.mark.parametrize("actions,nodes,depth,cpuct,c_pw", [(6, 300, 16, 1.5, 1.0), (225, 2000, 8, 1.5, 0.0),
                                                            (256, 600, 4, 0.7, 2.0), (3, 4000, 64, 1.0, 0.5),
                                                            (8, 1024, 24, 1.2, 1.0), (8, 1025, 24, 1.2, 1.0)])
def test_single_traversal_matches_oracle_exactly(actions, nodes, depth, cpuct, c_pw):
    """One traversal per tree is deterministic: every array must equal the oracle's, over several select/backup
    rounds on the same trees (the statistics drift apart as soon as one score comparison differs).  (A single traversal's claims
    are plain stores, whatever the size of the tree; up to 8192 edge slots, on either side of which the last two cases
    are, several would keep theirs in LDS.)"""
    rng = np.random.default_rng(actions * 1000 + nodes)
    case = pc.random_forest(rng, trees=64, nodes=nodes, actions=actions, warps=1, path_depth=depth)
    h = copy.deepcopy(case)
    r = HipRunner()
    for rnd in range(6):
        got = r.select(case if rnd == 0 else to_host(r.d), cpuct=cpuct, c_pw=c_pw)
        po.select(h, cpuct=cpuct, c_pw=c_pw)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        values = rng.uniform(-1, 1, h["out_path"].shape).astype(np.float32)
        got = r.backup(values)
        po.backup(h, values)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        assert pc.inflight_sum(got) == 0


@pytest.mark.parametrize("actions,nodes,hubs,claims,cpuct,c_pw,soft", [(256, 1200, 2, 0.05, 1.5, 0.0, 0), (193, 1200, 4, 0.3, 1.0, 16.0, 1),
                                                                      (129, 300, 1, 0.3, 0.5, 0.0, 0), (65, 300, 8, 0.05, 4.0, 2.0, 1),
                                                                      (225, 40, 1, 0.0, 0.0, 100.0, 0)])
def test_wide_nodes_with_claims_in_flight_match_oracle_exactly(actions, nodes, hubs, claims, cpuct, c_pw, soft):
    """As above on trees whose top levels fill two to four 64-edge slices, with random statistics, repeated priors and
    claims already held on some edges (so the scores see virtual loss)."""
    rng = np.random.default_rng(actions * 1000 + nodes)
    case = pc.wide_forest(rng, trees=32, nodes=nodes, actions=actions, warps=1, path_depth=12, hubs=hubs, claims=claims)
    h = copy.deepcopy(case)
    r = HipRunner()
    for rnd in range(4):
        got = r.select(case if rnd == 0 else to_host(r.d), cpuct=cpuct, c_pw=c_pw, soft_winner=soft)
        po.select(h, cpuct=cpuct, c_pw=c_pw, soft_winner=soft)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        values = rng.uniform(-1, 1, h["out_path"].shape).astype(np.float32)
        got = r.backup(values)
        po.backup(h, values)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)


@pytest.mark.parametrize("actions,nodes,depth,claims,cpuct,c_pw,soft", [
    (256, 30, 40, 0.1, 1.5, 0.0, 0), (256, 32, 64, 0.3, 0.5, 0.0, 1), (256, 33, 40, 0.1, 1.5, 0.0, 0), (193, 42, 100, 0.1, 1.0, 0.0, 0), (192, 42, 40, 0.0, 0.5, 2.0, 0),
    (129, 63, 200, 0.05, 1.5, 0.0, 1), (128, 64, 40, 0.3, 0.2, 1.2, 0), (65, 126, 64, 0.1, 1.5, 0.0, 0), (64, 128, 40, 0.1, 1.0, 0.0, 1), (64, 129, 40, 0.1, 1.0, 0.0, 0),
    (5, 3, 90, 0.0, 1.0, 0.0, 0)])
def test_single_traversals_of_recurrent_trees_match_oracle_exactly(actions, nodes, depth, claims, cpuct, c_pw, soft):
    """One traversal a tree on few nodes of one to four 64-edge slices, with claims already held, some of them on the edges
    that win; paths come back to edges that they hold a claim on, and some end at an edge that leads nowhere and give all of
    it back.  nodes * edges lies on both sides of 8192, which makes no difference to a single traversal (its claims are
    plain stores)."""
    rng = np.random.default_rng(actions * 1000 + nodes)
    case = pc.recurrent_forest(rng, trees=48, nodes=nodes, actions=actions, path_depth=depth, claims=claims, dead_ends=1.0 / min(depth, actions))
    h = copy.deepcopy(case)
    r = HipRunner()
    again = given_back = 0
    for rnd in range(4):
        got = r.select(case if rnd == 0 else to_host(r.d), cpuct=cpuct, c_pw=c_pw, soft_winner=soft)
        po.select(h, cpuct=cpuct, c_pw=c_pw, soft_winner=soft)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        for t in range(48):
            path = h["out_path"][t, 0, :max(0, h["out_len"][t, 0] - 1)]
            again += len(set(path.tolist())) < len(path)
            given_back += pc.decode(h["out_selected"][t, 0])[0] == pc.INVALID
        values = (np.floor(rng.uniform(-64, 64, h["out_path"].shape)) / 64).astype(np.float32)
        got = r.backup(values)
        po.backup(h, values)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
    assert given_back > 0 and (again > 0 or c_pw > 0)   # (with widening the paths are short)


@pytest.mark.parametrize("trees,actions,nodes,depth,warps,counted", [
    (4096, 9, 10, 128, 1, True), (1030, 64, 65, 512, 1, True), (1024, 90, 91, 130, 8, True), (4096, 20, 21, 70, 3, True), (600, 33, 34, 130, 16, True),
    (16, 64, 65, 300, 4, False), (4095, 9, 10, 128, 1, False), (8, 90, 92, 200, 16, False)])
def test_backup_of_long_paths_matches_oracle(trees, actions, nodes, depth, warps, counted):
    """Paths that come back to the nodes of a small tree, longer than a wavefront, by one to sixteen traversals; those that give way or end
    nowhere hold nothing.  On either side of where the backup may count in LDS what was passed (`counted`; it does for trees whose paths
    are long).  Values are multiples of 1/64
    small enough for their sums to be exact, so that every order of adding them gives the same."""
    from mcts_numba_cuda_amd import puct
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    assert counted == (nodes * actions <= 8192 and depth >= nodes and 40 * warps * depth >= nodes * actions and trees * warps * depth >= 1 << 19)
    rng = np.random.default_rng(trees + actions * 1000 + warps)
    case = pc.recurrent_forest(rng, trees=trees, nodes=nodes, actions=actions, path_depth=depth, claims=0.1, dead_ends=0.5 / depth)
    case["out_selected"], case["out_len"] = np.zeros((trees, warps), np.int32), np.zeros((trees, warps), np.int32)
    case["out_path"] = np.full((trees, warps, depth), -1, np.int32)
    r = HipRunner()
    for rnd, with_values in enumerate((True, False)):
        before = int((case if rnd == 0 else h)["edge_inflight"].sum())
        h = r.select(case if rnd == 0 else h, cpuct=1.5, c_pw=0.0, soft_winner=rnd)
        kinds = (h["out_selected"] >> 22) & 7
        holding = (kinds == pc.EXPAND) | (kinds == pc.TERMINAL_KIND) | (kinds == pc.DEPTH_LIMIT)
        assert holding.any() and np.all(h["out_len"][~holding] == 0) and h["out_len"].max() > 65
        assert int(h["edge_inflight"].sum()) - before == int((h["out_len"][holding] - 1).sum())   # (what gave way has taken all of it back)
        values = (np.floor(rng.uniform(-64, 64, h["out_path"].shape)) / 64).astype(np.float32) if with_values else None
        got = r.backup(values)
        at_nodes = copy.deepcopy(h)
        po.backup(h, values)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        # the same paths, as selections with node-level virtual loss report them
        del at_nodes["edge_inflight"]
        at_nodes["node_inflight"] = rng.integers(0, 1000, (trees, nodes)).astype(np.int32)
        at_nodes["out_selected"] = np.where(holding, at_nodes["out_selected"] & ((1 << 25) - 1), 0x3FFF).astype(np.int32)
        d = to_device(at_nodes)
        values = (np.floor(rng.uniform(-64, 64, h["out_path"].shape)) / 64).astype(np.float32)
        puct.launch_node_backup(d, DeviceArray(values))
        synchronize()
        got = to_host(d)
        po.backup(at_nodes, values, node_level=True)
        for k in at_nodes:
            assert np.array_equal(got[k], at_nodes[k], equal_nan=True), (rnd, k)


@pytest.mark.parametrize("trees,actions,nodes,depth,warps", [(16390, 9, 10, 40, 1), (8197, 20, 21, 70, 1), (2050, 90, 91, 300, 1), (4101, 20, 21, 70, 2), (1367, 64, 65, 130, 3),
                                                             (1025, 30, 31, 100, 8), (530, 90, 91, 91, 16), (600, 8, 1024, 1024, 1), (64, 1, 8192, 8192, 1)])
def test_backup_of_short_and_long_paths_matches_oracle(trees, actions, nodes, depth, warps):
    """Where paths may be long, a tree is counted by the levels that its paths have together: trees on either side of that line (24 + nodes *
    actions / 128 levels), with paths of no, one and two levels and of all that there is room for, next to each other, and numbers of
    trees that are no multiple of a workgroup's.  Values and sums are multiples of 1/64, exact in every order of adding them."""
    from mcts_numba_cuda_amd import puct
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    rng = np.random.default_rng(trees + actions)
    line, shape = 24 + nodes * actions // 128, (trees, nodes, actions)
    d = {"edge_child": rng.integers(-1, nodes + 1, shape).astype(np.int32), "edge_w": np.zeros(shape, np.float32), "edge_n": rng.integers(0, 50, shape).astype(np.int32),
         "edge_inflight": rng.integers(0, 50, shape).astype(np.int32), "node_expand_inflight": rng.integers(0, 9, shape[:2]).astype(np.int32),
         "node_count": rng.integers(nodes // 2, nodes + 1, trees).astype(np.int32)}
    # how the levels of a tree are shared out among its traversals: evenly, or all to the last
    levels = rng.choice([0, 1, 2, line - 1, line, line + 1, depth, warps * depth], trees)
    each = np.minimum(np.diff(np.floor(levels[:, None] * np.arange(warps + 1) / warps).astype(np.int64), axis=1), depth)
    alone = rng.random(trees) < 0.3
    each[alone] = 0
    each[alone, -1] = np.minimum(levels[alone], depth)
    kind = np.where(each > 0, rng.choice([pc.EXPAND, pc.TERMINAL_KIND, pc.DEPTH_LIMIT], each.shape), rng.choice([pc.INVALID, pc.BUSY, pc.EXPAND, pc.TERMINAL_KIND], each.shape))
    d["out_selected"] = ((kind << 22) | rng.integers(0, nodes, each.shape)).astype(np.int32)
    d["out_len"] = np.where((kind == pc.INVALID) | (kind == pc.BUSY), 0, each + 1).astype(np.int32)
    d["out_path"] = (rng.integers(0, nodes, (trees, warps, depth)) << 8 | rng.integers(0, actions, (trees, warps, depth))).astype(np.int32)
    d["out_path"][rng.random(d["out_path"].shape) < 0.01] = -1
    assert depth >= nodes and nodes * actions <= 8192 and 40 * warps * depth >= nodes * actions and trees * warps * depth >= 1 << 19 and line <= warps * depth
    sums = each.sum(1)
    assert all(np.any(sums == n) for n in ((line - 1, line) if line <= depth else ()))
    for node_level in (False, True):
        h = copy.deepcopy(d)
        if node_level:
            del h["edge_inflight"]
            h["node_inflight"] = rng.integers(0, 999, (trees, nodes)).astype(np.int32)
            h["out_selected"] = np.where(kind == pc.BUSY, 0x3FFF, h["out_selected"]).astype(np.int32)
        for with_values in ((True,) if node_level else (True, False)):
            got = to_device(h)
            values = (np.floor(rng.uniform(-64, 64, h["out_path"].shape)) / 64).astype(np.float32) if with_values else None
            (puct.launch_node_backup if node_level else puct.launch_edge_backup)(got, None if values is None else DeviceArray(values))
            synchronize()
            po.backup(h, values, node_level=node_level)
            got = to_host(got)
            for k in h:
                assert np.array_equal(got[k], h[k]), (node_level, with_values, k)


def launch_times(launch, launches=60, rounds=7):
    """Fastest of `rounds` mean times of a launch, in us."""
    from mcts_numba_cuda_amd.hipmem import Event
    best = np.inf
    for _ in range(rounds):
        start, end = Event(), Event()
        start.record()
        for _ in range(launches):
            launch()
        end.record()
        synchronize()
        best = min(best, 1e3 * start.elapsed_ms(end) / launches)
    return best


def test_backup_of_short_paths_does_not_pay_for_the_room_that_they_have():
    """Paths of one and two levels where 512 would fit, which is more than the trees have nodes, and where 64 would, which is less: 7.0 and 5.2 us;
    when all trees of the first kind were counted it took 26."""
    from mcts_numba_cuda_amd import puct
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    trees, nodes, actions = 16384, 65, 64
    rng = np.random.default_rng(3)
    d = {k: DeviceArray(np.zeros((trees, nodes, actions), t)) for k, t in (("edge_w", np.float32), ("edge_n", np.int32), ("edge_inflight", np.int32))}
    d.update({"node_expand_inflight": DeviceArray(np.zeros((trees, nodes), np.int32)), "node_count": DeviceArray(np.full(trees, nodes, np.int32)),
              "out_selected": DeviceArray(np.full((trees, 1), pc.TERMINAL_KIND << 22, np.int32)), "out_len": DeviceArray(rng.integers(2, 4, (trees, 1)).astype(np.int32))})
    path = (rng.integers(0, nodes, (trees, 1, 512)) << 8 | rng.integers(0, actions, (trees, 1, 512))).astype(np.int32)
    roomy, tight = (dict(d, out_path=DeviceArray(path[:, :, :n])) for n in (512, 64))
    launch, fields = puct._lib().puct_edge_backup_launch, ("edge_w", "edge_n", "edge_inflight", "node_expand_inflight", "node_count", "out_selected", "out_path", "out_len")
    times = []
    for x in (roomy, tight):   # (the C function itself: the arguments' checks take longer than the launch)
        arguments = (1, *(x[k].data_ptr() for k in fields), None, trees, nodes, actions, 1, x["out_path"].shape[2], None)
        times.append(launch_times(lambda: launch(*arguments)))
    assert times[0] < 2.5 * times[1], times


@pytest.mark.parametrize("actions,nodes,depth,warps", [
    (256, 32, 200, 8), (256, 33, 200, 8), (193, 42, 150, 16), (193, 43, 150, 16), (129, 63, 200, 3), (129, 64, 200, 3), (65, 126, 140, 16), (65, 127, 140, 16), (64, 128, 200, 2),
    (64, 129, 200, 2), (192, 20, 128, 16), (128, 70, 90, 5), (256, 20, 150, 17), (193, 60, 130, 24), (65, 40, 200, 33), (5, 9, 90, 16), (100, 80, 120, 8),
    (256, 90, 100, 8), (193, 140, 200, 20)])
def test_settled_traversals_match_oracle_exactly(actions, nodes, depth, warps):
    """Several traversals a tree, where their order does not matter: every array must equal the oracle's.  Nodes of one to four 64-edge slices; up to
    16 traversals with claims in LDS (nodes * edges <= 8192) or in memory, and more than 16, in several workgroups.  Claims are lost to others and
    taken again, paths are longer than a wavefront, and those that end nowhere are given back."""
    trees = 24
    rng = np.random.default_rng(actions * 1000 + nodes + warps)
    case = pc.settled_forest(rng, trees=trees, nodes=nodes, actions=actions, warps=warps, path_depth=depth)
    h, other = copy.deepcopy(case), copy.deepcopy(case)
    other["edge_inflight"][:] = rng.integers(0, 2 * warps, other["edge_inflight"].shape)
    po.select(other, cpuct=1e-3, c_pw=0.0, soft_winner=1)
    r = HipRunner()
    for rnd in range(2):
        got = r.select(case if rnd == 0 else to_host(r.d), cpuct=1e-3, c_pw=0.0, soft_winner=1)
        po.select(h, cpuct=1e-3, c_pw=0.0, soft_winner=1)
        if rnd == 0:   # (whatever is claimed already)
            assert all(np.array_equal(h[k], other[k]) for k in ("out_selected", "out_path", "out_len"))
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
    kinds, reasons = (h["out_selected"] >> 22) & 7, (h["out_selected"] >> 25) & 0x3F
    assert {pc.INVALID, pc.TERMINAL_KIND} <= set(kinds.ravel().tolist()) <= {pc.INVALID, pc.TERMINAL_KIND, pc.DEPTH_LIMIT}
    given_back = (kinds == pc.INVALID) & np.isin(reasons, (11, 14, 15))
    assert set(reasons[given_back].tolist()) == {11, 14, 15} and np.any((case["edge_inflight"] > 0) & (h["edge_inflight"] > case["edge_inflight"] + 1))
    levels = (h["out_path"] >= 0).sum(axis=2)
    assert levels.max() > 64 and (min(nodes, depth) <= 66 or levels[given_back].max() > 64)
    got = r.backup(None)
    po.backup(h, None)
    for k in h:
        assert np.array_equal(got[k], h[k], equal_nan=True), k


@pytest.mark.parametrize("trees,warps,soft", [(16, 8, 0), (16, 16, 0), (4, 40, 0), (16, 16, 1), (128, 4, 0)])
def test_concurrent_traversals_keep_invariants(trees, warps, soft):
    rng = np.random.default_rng(trees * 100 + warps)
    case = pc.random_forest(rng, trees=trees, nodes=400, actions=16, warps=warps, path_depth=12)
    n_before, w_before = case["edge_n"].copy(), case["edge_w"].copy()
    r = HipRunner()
    h = r.select(case, cpuct=1.5, c_pw=1.0, soft_winner=soft)
    assert pc.inflight_nonnegative(h)
    kinds = (h["out_selected"] >> 22) & 7
    assert np.all(np.isin(kinds, (pc.EXPAND, pc.TERMINAL_KIND, pc.DEPTH_LIMIT, pc.BUSY)))
    if soft:
        assert not np.any((kinds == pc.BUSY) & (((h["out_selected"] >> 25) & 0x3F) == 5))
    holding = (kinds != pc.BUSY)
    assert np.any(holding)
    assert np.all(h["out_len"][~holding] == 0)
    assert int(h["edge_inflight"].sum()) == int((h["out_len"][holding] - 1).sum())
    assert int(h["node_expand_inflight"].sum()) == int((kinds == pc.EXPAND).sum())
    # expansion slots of one node are distinct and start at its current child count
    for t in range(trees):
        seen = set()
        for w in range(warps):
            k, slot, node = pc.decode(h["out_selected"][t, w])
            if k == pc.EXPAND:
                assert (node, slot) not in seen and slot >= h["node_expanded"][t, node]
                seen.add((node, slot))
    # every recorded path is a chain of existing edges from the root to the selected node
    for t in range(trees):
        for w in range(warps):
            if not holding[t, w]:
                continue
            node = 0
            for dd in range(h["out_len"][t, w] - 1):
                enc = int(h["out_path"][t, w, dd])
                assert enc >> 8 == node and (enc & 0xFF) < h["node_expanded"][t, node]
                node = int(h["edge_child"][t, node, enc & 0xFF])
            assert node == pc.decode(h["out_selected"][t, w])[2]
    values = np.full(h["out_path"].shape, 0.5, np.float32)
    h2 = r.backup(values)
    assert pc.inflight_sum(h2) == 0 and pc.inflight_nonnegative(h2)
    added = h2["edge_n"] - n_before
    assert int(added.sum()) == int((h["out_len"][holding] - 1).sum())
    assert np.allclose(h2["edge_w"] - w_before, 0.5 * added, atol=1e-3)


def test_node_level_backup_known_answer():
    """src/puct/test_puct_gpu_v2.py:1085-1119 through puct_node_backup_launch."""
    from mcts_numba_cuda_amd import puct
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    h = pc.make_case(nodes=3, actions=4, path_depth=4)
    h["edge_child"][0, 0, :2] = (1, 2)
    h["edge_n"][0, 0, :2] = 1
    h["node_inflight"] = np.zeros((1, 3), np.int32)
    h["node_inflight"][0, 2] = 1
    h["node_expand_inflight"][0, 2] = 1
    h["out_selected"][0, 0] = (pc.EXPAND << 22) | 2
    h["out_path"][0, 0, 0] = 1
    h["out_len"][0, 0] = 2
    values = np.zeros((1, 1, 4), np.float32)
    values[0, 0, 0] = 0.7
    d = to_device(h)
    puct.launch_node_backup(d, DeviceArray(values))
    synchronize()
    g = to_host(d)
    assert int(g["node_inflight"].sum()) == 0 and int(g["node_expand_inflight"].sum()) == 0
    assert g["edge_n"][0, 0, 1] == 2 and g["edge_w"][0, 0, 1] == np.float32(0.7)
    ref = copy.deepcopy(h)
    po.backup(ref, values, node_level=True)
    for k in ref:
        assert np.array_equal(g[k], ref[k]), k


def test_launch_errors_are_reported():
    from mcts_numba_cuda_amd import puct
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    case = pc.make_case(nodes=2, actions=4, warps=1, path_depth=2)
    d = to_device(case)
    d["edge_prior"] = DeviceArray(case["edge_prior"].astype(np.float64))
    with pytest.raises(ValueError):
        puct.launch_select(d)
    d = to_device(case)
    d["out_selected"] = DeviceArray(np.zeros((1, 0), np.int32))
    d["out_len"] = DeviceArray(np.zeros((1, 0), np.int32))
    d["out_path"] = DeviceArray(np.zeros((1, 0, 2), np.int32))
    with pytest.raises(RuntimeError, match="launch failed"):
        puct.launch_select(d)           # zero traversals: the runtime rejects the empty launch, as CUDA does
    assert isinstance(puct._lib().puct_cpp_cuda_error_string(0), bytes)
