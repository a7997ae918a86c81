"""PUCT selection with node-level virtual loss (puct_node_select_preclaim_launch, puct_node_select_winner_recalc_launch)
and its backup through the C ABI of libpuct_hip.so on the GPU: the reference's known answers, bit-exact agreement with
the sequential oracle wherever a launch is deterministic (one traversal per tree), and the invariants every interleaving
satisfies where it is not."""
import copy

import numpy as np
import pytest

import puct_node_cases as nc
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


class HipRunner(nc.Runner):
    def select(self, case, variant, **params):
        from mcts_numba_cuda_amd import puct
        self.d = to_device(case)
        puct.launch_node_select(self.d, variant=variant, **params)
        synchronize()
        return to_host(self.d)

    def backup(self, values):
        from mcts_numba_cuda_amd import puct
        from mcts_numba_cuda_amd.hipmem import DeviceArray
        puct.launch_node_backup(self.d, DeviceArray(values))
        synchronize()
        return to_host(self.d)


@pytest.mark.parametrize("variant", nc.VARIANTS)
@pytest.mark.parametrize("case", nc.ALL_CASES, ids=lambda f: f.__name__)
def test_known_answers(case, variant):
    case(HipRunner(), variant)


@pytest.mark.parametrize("variant", nc.VARIANTS)
@pytest.mark.parametrize("actions,nodes,depth,cpuct,c_pw", [(6, 300, 16, 1.5, 1.0), (225, 2000, 8, 1.5, 0.0),
                                                            (256, 600, 4, 0.7, 2.0), (3, 4000, 64, 1.0, 0.5),
                                                            (5, 16384, 24, 1.2, 1.0), (5, 16385, 24, 1.2, 1.0)])
def test_single_traversal_matches_oracle_exactly(actions, nodes, depth, cpuct, c_pw, variant):
    """One traversal per tree is deterministic: every array must equal the oracle's, over several select/backup rounds on
    the same trees (the statistics drift apart as soon as one score comparison differs).  In every other round the
    claims of the selection are left in place for the next one, so that the kernels also score against virtual visits.
    (A tree's counters are in LDS during a launch up to 200 * path_depth nodes for every 64 edges, here 300 and 4000 nodes,
    and in device memory beyond; the test below is about that line.)"""
    rng = np.random.default_rng(actions * 1000 + nodes)
    case = nc.random_forest(rng, trees=64, nodes=nodes, actions=actions, warps=1, path_depth=depth)
    h = copy.deepcopy(case)
    r = HipRunner()
    for rnd in range(8):
        got = r.select(case if rnd == 0 else to_host(r.d), variant, cpuct=cpuct, c_pw=c_pw)
        po.node_select(h, cpuct=cpuct, c_pw=c_pw, variant=variant)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        if rnd % 2 == 1:
            continue          # keep this round's claims (expansion tickets included) for the next selection
        values = rng.uniform(-1, 1, h["out_path"].shape).astype(np.float32)
        got = r.backup(values)
        po.backup(h, values, node_level=True)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)


@pytest.mark.parametrize("variant", nc.VARIANTS)
@pytest.mark.parametrize("actions,nodes,depth", [(5, 800, 4), (5, 801, 4), (64, 1000, 5), (64, 1001, 5), (65, 800, 2), (65, 801, 2), (129, 1200, 2), (129, 1201, 2), (256, 1600, 2), (256, 1601, 2),
                                                 (5, 16384, 82), (5, 16384, 81), (5, 16385, 82), (3, 16384, 1024), (3, 16385, 1024)])
def test_single_traversals_on_either_side_of_counters_in_lds(actions, nodes, depth, variant):
    """Counters in LDS up to 200 * path_depth nodes for every 64 edges and up to 16384 nodes, in memory beyond: as above, with visits already on some of
    the nodes, those beyond the last among them, which nobody may change."""
    rng = np.random.default_rng(actions * 1000 + nodes + depth)
    trees = 3 if nodes > 2000 else 8
    case = nc.random_forest(rng, trees=trees, nodes=nodes, actions=actions, warps=1, path_depth=depth)
    case["node_inflight"][:] = np.where(rng.random(case["node_inflight"].shape) < 0.5, rng.integers(1, 5, case["node_inflight"].shape), 0)
    case["node_count"][0] = nodes if nodes <= 16384 else 16384
    h = copy.deepcopy(case)
    r = HipRunner()
    for rnd in range(4):
        got = r.select(case if rnd == 0 else to_host(r.d), variant, cpuct=1.2, c_pw=1.0)
        po.node_select(h, cpuct=1.2, c_pw=1.0, variant=variant)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        values = rng.uniform(-1, 1, h["out_path"].shape).astype(np.float32)
        got = r.backup(values)
        po.backup(h, values, node_level=True)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)


@pytest.mark.parametrize("actions,nodes,depth,warps", [(64, 130, 200, 2), (256, 90, 120, 16), (193, 100, 120, 7), (129, 70, 90, 3), (65, 5003, 90, 2), (9, 12007, 70, 16), (9, 16384, 70, 11),
                                                       (9, 16385, 70, 4), (256, 90, 100, 17), (193, 40, 100, 24), (129, 140, 200, 33), (64, 80, 100, 20)])
def test_settled_preclaims_match_oracle_exactly(actions, nodes, depth, warps):
    """Several traversals a tree, where their order does not matter: every array must equal the oracle's, with up to 16 traversals (counters in LDS up to
    16384 nodes, copied eight words at a time and then one by one: neither 5003 nor 12007 nor 16384 is a multiple of what that takes) and
    more of them (counters in memory).  Visits are on some of the nodes beforehand, most of which nobody comes to."""
    rng = np.random.default_rng(actions * 1000 + nodes + warps)
    case = nc.settled_forest(rng, trees=4 if nodes > 2000 else 24, nodes=nodes, actions=actions, warps=warps, path_depth=depth)
    if nodes > 16384:
        case["node_count"][:] = 16384
    h, other = copy.deepcopy(case), copy.deepcopy(case)
    other["node_inflight"][:] = rng.integers(0, 2 * warps, other["node_inflight"].shape)
    po.node_select(other, cpuct=1e-3, c_pw=0.0, variant="preclaim")
    r = HipRunner()
    for rnd in range(2):
        got = r.select(case if rnd == 0 else to_host(r.d), "preclaim", cpuct=1e-3, c_pw=0.0)
        po.node_select(h, cpuct=1e-3, c_pw=0.0, variant="preclaim")
        if rnd == 0:   # (whatever is claimed already)
            assert all(np.array_equal(h[k], other[k]) for k in ("out_selected", "out_path", "out_len"))
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
    assert (h["out_path"] >= 0).sum(axis=2).max() > 64 or nodes > 2000
    got = r.backup(nc.zeros_like_path(h))
    po.backup(h, nc.zeros_like_path(h), node_level=True)
    for k in h:
        assert np.array_equal(got[k], h[k], equal_nan=True), k


@pytest.mark.parametrize("variant", nc.VARIANTS)
@pytest.mark.parametrize("nodes,warps", [(5003, 2), (5003, 3), (12007, 16), (16384, 16), (4099, 17)])
def test_counters_of_nodes_that_nobody_comes_to_stay(nodes, warps, variant):
    """Several traversals, whose claims depend on each other, on trees of several thousand nodes with visits on them: what has been added to the counters
    is one for every path edge, on the node it leads to, and nothing on any other node, whoever keeps them."""
    rng = np.random.default_rng(nodes + warps)
    case = nc.random_forest(rng, trees=4, nodes=nodes, actions=12, warps=warps, path_depth=24)
    case["node_inflight"][:] = rng.integers(0, 4, case["node_inflight"].shape)
    h = HipRunner().select(case, variant, cpuct=1.5, c_pw=0.6)
    kinds = h["out_selected"] >> 22
    assert np.any(kinds != nc.INVALID) and np.all(h["out_len"][kinds == nc.INVALID] == 0)
    want = case["node_inflight"].copy()
    for t, w in zip(*np.nonzero(kinds != nc.INVALID)):
        for enc in h["out_path"][t, w, :h["out_len"][t, w] - 1]:
            want[t, case["edge_child"][t, enc >> 8, enc & 0xFF]] += 1
    assert np.array_equal(h["node_inflight"], want)


@pytest.mark.parametrize("variant", nc.VARIANTS)
@pytest.mark.parametrize("actions,nodes,hubs,visits,cpuct,c_pw", [(256, 1200, 2, 0.05, 1.5, 0.0), (193, 1200, 4, 0.3, 1.0, 16.0),
                                                                 (129, 300, 1, 0.3, 0.5, 0.0), (65, 300, 8, 0.05, 4.0, 2.0),
                                                                 (225, 40, 1, 0.0, 0.0, 100.0)])
def test_wide_nodes_with_virtual_visits_match_oracle_exactly(actions, nodes, hubs, visits, cpuct, c_pw, variant):
    """As above on trees whose top levels fill two to four 64-edge slices, with random statistics, repeated priors,
    virtual visits already on some nodes and some expanded edges that lead nowhere."""
    rng = np.random.default_rng(actions * 1000 + nodes)
    case = nc.wide_forest(rng, trees=32, nodes=nodes, actions=actions, warps=1, path_depth=12, hubs=hubs, visits=visits)
    h = copy.deepcopy(case)
    r = HipRunner()
    for rnd in range(4):
        got = r.select(case if rnd == 0 else to_host(r.d), variant, cpuct=cpuct, c_pw=c_pw)
        po.node_select(h, cpuct=cpuct, c_pw=c_pw, variant=variant)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)
        values = rng.uniform(-1, 1, h["out_path"].shape).astype(np.float32)
        got = r.backup(values)
        po.backup(h, values, node_level=True)
        for k in h:
            assert np.array_equal(got[k], h[k], equal_nan=True), (rnd, k)


@pytest.mark.parametrize("variant", nc.VARIANTS)
@pytest.mark.parametrize("trees,warps", [(16, 8), (16, 16), (4, 40), (128, 4)])
def test_concurrent_traversals_keep_invariants(trees, warps, variant):
    rng = np.random.default_rng(trees * 100 + warps)
    case = nc.random_forest(rng, trees=trees, nodes=400, actions=16, warps=warps, path_depth=12)
    n_before, w_before = case["edge_n"].copy(), case["edge_w"].copy()
    r = HipRunner()
    h = r.select(case, variant, cpuct=1.5, c_pw=1.0)
    assert nc.inflight_nonnegative(h)
    kinds = h["out_selected"] >> 22
    assert np.all(np.isin(kinds, (nc.INVALID, nc.EXPAND, nc.TERMINAL_KIND, nc.DEPTH_LIMIT)))
    holding = kinds != nc.INVALID
    assert np.any(holding)
    assert np.all(h["out_len"][~holding] == 0) and np.all(h["out_selected"][~holding] == nc.PACKED_INVALID)
    assert int(h["node_expand_inflight"].sum()) == int((kinds == nc.EXPAND).sum())
    # expansion slots of one node are distinct and start at its current child count
    for t in range(trees):
        seen = set()
        for w in range(warps):
            k, slot, node = nc.decode(h["out_selected"][t, w])
            if k == nc.EXPAND:
                assert (node, slot) not in seen and slot >= h["node_expanded"][t, node]
                seen.add((node, slot))
    # every recorded path is a chain of existing edges from the root to the selected node, and the claims that are left
    # are exactly one per path edge, on the node the edge leads to (every passing claim of a preclaim was given back)
    want = np.zeros_like(h["node_inflight"])
    for t, w in zip(*np.nonzero(holding)):
        node = 0
        for dd in range(h["out_len"][t, w] - 1):
            enc = int(h["out_path"][t, w, dd])
            assert enc >> 8 == node and (enc & 0xFF) < h["node_expanded"][t, node]
            node = int(h["edge_child"][t, node, enc & 0xFF])
            assert 0 <= node < h["node_count"][t]
            want[t, node] += 1
        assert node == nc.decode(h["out_selected"][t, w])[2]
    assert np.array_equal(want, h["node_inflight"])
    values = np.full(h["out_path"].shape, 0.5, np.float32)
    h2 = r.backup(values)
    assert nc.inflight_sum(h2) == 0 and nc.inflight_nonnegative(h2)
    added = h2["edge_n"] - n_before
    assert int(added.sum()) == int((h["out_len"][holding] - 1).sum())
    assert np.allclose(h2["edge_w"] - w_before, 0.5 * added, atol=1e-3)


@pytest.mark.parametrize("variant", nc.VARIANTS)
def test_deep_wide_shape_of_the_reference_benchmark(variant):
    """The reference's large-scale select benchmark at a size that runs in a moment (src/puct/test_puct_gpu_v2.py:
    1802-1915, shape "wide" of :109-143): every node has `actions` children on the same `actions` nodes, equal priors,
    c_pw = 0, eight traversals per tree walk `depth` levels to the depth limit; its own criterion: full-length paths,
    some valid selections, nothing in flight after the backup."""
    trees, actions, depth, warps = 64, 64, 128, 8
    c = nc.make_case(trees=trees, nodes=actions + 1, actions=actions, warps=warps, path_depth=depth)
    c["node_expanded"][:] = actions
    c["edge_child"][:] = np.arange(1, actions + 1, dtype=np.int32)
    c["edge_n"][:] = 1
    r = HipRunner()
    h = r.select(c, variant, cpuct=1.0, c_pw=0.0)
    kinds = h["out_selected"] >> 22
    assert np.all(kinds == nc.DEPTH_LIMIT) and np.all(h["out_len"] == depth + 1)
    assert int(h["node_inflight"].sum()) == trees * warps * depth and nc.inflight_nonnegative(h)
    h2 = r.backup(nc.zeros_like_path(h))
    assert nc.inflight_sum(h2) == 0 and int(h2["edge_n"].sum()) == int(c["edge_n"].sum()) + trees * warps * depth


@pytest.mark.parametrize("variant", nc.VARIANTS)
def test_a_single_traversals_counters_cost_no_jump(variant):
    """64 trees of 700 nodes with 16 edges, one traversal of 43 and of 44 levels: 29 and 30 us (winner-recalc 39 and 40).
    When a tree of more than 16 * path_depth nodes had its counters in memory, 43 levels took 58 and 62."""
    from mcts_numba_cuda_amd import puct
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    from test_gpu_puct import launch_times
    trees, actions, nodes = 64, 16, 700
    launch = {"preclaim": puct._lib().puct_node_select_preclaim_launch, "winner_recalc": puct._lib().puct_node_select_winner_recalc_launch}[variant]
    times = []
    for depth in (43, 44):
        c = nc.make_case(trees=trees, nodes=nodes, actions=actions, warps=1, path_depth=depth)
        c["node_expanded"][:] = actions
        c["edge_child"][:] = np.arange(1, actions + 1, dtype=np.int32)
        c["edge_n"][:] = 1
        d = to_device(c)
        arguments = (1.0, 0.0, 0.5, *(d[k].data_ptr() for k in ("edge_child", "edge_prior", "edge_w", "edge_n", "node_inflight", "node_expand_inflight", "node_expanded", "node_count",
                                                             "out_selected", "out_path", "out_len")), trees, nodes, actions, 1, depth, None)
        times.append(launch_times(lambda: launch(*arguments)))
        h = to_host(d)
        assert np.all(h["out_len"] == depth + 1)
    assert times[0] < 1.3 * times[1], times


def test_launch_errors_are_reported():
    from mcts_numba_cuda_amd import puct
    from mcts_numba_cuda_amd.hipmem import DeviceArray
    case = nc.make_case(nodes=2, actions=4, warps=1, path_depth=2)
    d = to_device(case)
    with pytest.raises(ValueError, match="variant"):
        puct.launch_node_select(d, variant="native")
    d["node_inflight"] = DeviceArray(case["node_inflight"].astype(np.int64))
    with pytest.raises(ValueError):
        puct.launch_node_select(d)
