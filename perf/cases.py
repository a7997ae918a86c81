"""The work that a user of this package has it do, as cases that can be timed and compared.

A case is one call of a public entry point as a program makes it: a search of one position (`MCTSNC.run`), of many
positions in one pass (`run_batch`), one selection and backup over a forest of PUCT trees (`launch_select` /
`launch_node_select` and the backups), or one search of the Gomoku PUCT loop (`PUCTGomoku.run`).  Searches read back what a
player reads after a move: the best action, the table of root actions and the statistics of the trees.

Search budgets are step counts, so that the same inputs are the same work: with a seed, a search is a pure function of
its root and of the random streams that its engine carries from search to search."""
import math

import numpy as np
import torch   # (before the package: torch brings its own copy of the HIP runtime, and the first one loaded serves both)

from mcts_numba_cuda_amd import C4, MCTSNC, puct, run_batch
from mcts_numba_cuda_amd.puct_gomoku import PUCTGomoku

VARIANTS = ("ocp_thrifty", "ocp_prodigal", "acp_thrifty", "acp_prodigal")
DEVICE = "cuda:0"


def _search(name, game, rows, columns, stones_low, stones_high, variant, trees, playouts, steps, memory, searches=1):
    return dict(name=name, kind="search", game=game, rows=rows, columns=columns, stones_low=stones_low, stones_high=stones_high,
                variant=variant, trees=trees, playouts=playouts, steps=steps, memory=memory, searches=searches)


def _select(name, claims, shape, trees, nodes, edges, traversals, depth, rule="winner_recalc"):
    return dict(name=name, kind="select", claims=claims, shape=shape, trees=trees, nodes=nodes, edges=edges, traversals=traversals,
                depth=depth, rule=rule)


def listed():
    return [
        # a quick answer on a small budget: a weak opponent, a hint, the inner search of a larger program
        _search("c4_small", "c4", 6, 7, 6, 6, "ocp_thrifty", 1, 32, 100, 0.05),
        # the usual player of a Connect 4 match, on one middle-game position after the other
        _search("c4_match", "c4", 6, 7, 10, 20, "acp_prodigal", 4, 256, 5000, 2.0),
        # a long analysis of the opening: trees that grow to a hundred thousand nodes
        _search("c4_analysis", "c4", 6, 7, 0, 0, "acp_thrifty", 8, 256, 20000, 16.0),
        # as many trees as the class takes, voting on one position
        _search("c4_512_trees", "c4", 6, 7, 0, 8, "acp_prodigal", 512, 256, 500, 0.3),
        # the moves of many games that are played side by side
        _search("c4_64_games", "c4", 6, 7, 10, 20, "acp_prodigal", 4, 256, 2000, 0.06, searches=64),
        # the one-child player of a Gomoku match
        _search("gomoku_match", "gomoku", 15, 15, 0, 20, "ocp_thrifty", 4, 128, 2000, 4.0),
        # the same game by the all-children player: every step plays out all empty cells
        _search("gomoku_all_children", "gomoku", 15, 15, 12, 18, "acp_prodigal", 8, 128, 400, 2.0),
        # the full-size board
        _search("gomoku_19", "gomoku", 19, 19, 0, 40, "ocp_prodigal", 4, 128, 300, 2.0),
        # one small batch of trees between two evaluations of a network: a selection and its backup, over and over
        _select("puct_select_small", "edge", "forest", 16, 257, 64, 8, 32),
        # self-play with many games in flight, eight leaves a game and batch
        _select("puct_select_forest", "edge", "forest", 1024, 4097, 64, 8, 32),
        # deep recurrent trees, every path to the depth limit
        _select("puct_select_deep", "edge", "deep", 16384, 65, 64, 1, 512),
        # the whole loop on the device, with every traversal of a step reaching a leaf
        dict(name="puct_gomoku", kind="loop", rows=15, columns=15, stones_low=0, stones_high=10, trees=16, traversals=16, steps=1000,
             c_pw=16.0, nodes=32768, depth=64),
    ]


# ---- drawn cases -------------------------------------------------------------------------------------------------------
def _log_uniform(rng, low, high):
    return low * (high / low) ** rng.random()


def _log_int(rng, low, high):
    return min(high, max(low, int(round(_log_uniform(rng, low, high)))))


def _step_seconds(game, cells, actions, acp, trees, playouts):
    """About what a step of all `trees` takes at most, to keep a drawn case within the largest listed one."""
    if game == "c4":
        return max(6e-6, trees * actions * playouts / 9e9) if acp else max(5e-6, trees * playouts / 3e9)
    if acp:
        return 60e-6 + trees * cells * playouts / 8e8 * (cells / 225) ** 2.5 * max(1.0, 64 / playouts)
    return 70e-6 * (cells / 225) ** 2.2 * math.ceil(playouts / 128) * math.ceil(trees / 256)


def draw(rng):
    family = rng.choice(["c4", "c4", "c4_games", "gomoku", "gomoku", "gomoku_games", "select", "select", "loop"])
    if family == "loop":
        trees, traversals = _log_int(rng, 1, 32), rng.randint(1, 16)
        steps = _log_int(rng, 50, 2000)
        rows, columns = rng.randint(9, 16), rng.randint(9, 16)
        return dict(kind="loop", rows=rows, columns=columns, stones_low=0, stones_high=rng.randint(0, 20), trees=trees, traversals=traversals,
                    steps=steps, c_pw=rng.choice([1.0, 16.0]), nodes=min(1 << 20, traversals * steps + 2), depth=64)
    if family == "select":
        claims = rng.choice(["edge", "edge", "node"])
        rule = rng.choice(["winner_recalc", "preclaim"]) if claims == "node" else "winner_recalc"
        edges = _log_int(rng, 9, 256)
        if rng.random() < 0.3:   # deep recurrent trees
            case = _select("", claims, "deep", _log_int(rng, 16, 16384), edges + 1, edges, 1, _log_int(rng, 16, 512), rule)
        else:
            traversals = rng.randint(1, 16)
            fewest = max(4 * edges + 1, 800 * traversals // edges)
            case = _select("", claims, "forest", _log_int(rng, 4, 2048), _log_int(rng, fewest, 8192), edges, traversals, rng.randint(16, 64), rule)
        while case["trees"] * case["nodes"] * case["edges"] > 1.5e8:
            case["trees"] = case["trees"] // 2
        case.pop("name")
        return case
    searches = 1
    variant = rng.choice(VARIANTS)
    acp = variant.startswith("acp")
    playouts = rng.choice([32, 64, 128, 256])
    trees = rng.choice([1, 2, 4, 8])
    if family.startswith("c4"):
        game = "c4"
        rows, columns = rng.choice([(6, 7), (6, 7), (6, 7), (7, 8), (5, 6), (8, 7)])
        stones = rng.randint(0, 20)
        if family == "c4_games":
            searches = _log_int(rng, 2, 256)
        elif rng.random() < 0.4:
            trees = _log_int(rng, 1, 512)
    else:
        game = "gomoku"
        rows = columns = rng.choice([9, 11, 13, 15, 15, 15, 19])
        if rng.random() < 0.2:
            rows = min(22, rows + rng.randint(0, 4))
        stones = rng.randint(0, rows * columns // 6)
        if family == "gomoku_games":
            searches = _log_int(rng, 2, 64)
        elif rng.random() < 0.3:
            trees = _log_int(rng, 1, 64)
    actions = columns if game == "c4" else rows * columns
    per_step = _step_seconds(game, rows * columns, actions, acp, trees * searches, playouts)
    steps = min(20000, max(20, int(_log_uniform(rng, 3e-4, 0.15) / per_step)))
    while steps * per_step > 0.2 and trees * searches > 1:   # a few steps of very many trees would cost more than any listed case
        trees, searches = max(1, trees // 2), max(1, searches // 2)
        per_step = _step_seconds(game, rows * columns, actions, acp, trees * searches, playouts)
    per_state = (95 if game == "c4" else 5.1 * rows * columns) + 20
    memory = max(0.01, 1.2 * trees * (steps + 2) * actions * per_state / 2**30)
    memory = min(memory, 24.0 / searches)
    if rng.random() < 0.1:
        memory *= 0.3   # a pool that runs full before the search ends
    case = _search("", game, rows, columns, stones, stones, variant, trees, playouts, steps, memory, searches)
    case.pop("name")
    return case


# ---- inputs ------------------------------------------------------------------------------------------------------------
def _has_line(board, token, length):
    m, n = board.shape
    own = board == token
    for di, dj in ((0, 1), (1, 0), (1, 1), (1, -1)):
        h, w = m - di * (length - 1), n - abs(dj) * (length - 1)
        if h <= 0 or w <= 0:
            continue
        run = np.ones((h, w), bool)
        for k in range(length):
            j = k * dj if dj >= 0 else (length - 1 - k)
            run &= own[k * di:k * di + h, j:j + w]
        if run.any():
            return True
    return False


def _c4_root(rng, rows, columns, plies):
    """A position after `plies` uniformly random legal moves, none of which ended the game."""
    while True:
        board, fills, turn = np.zeros((rows, columns), np.int8), np.zeros(columns, np.int8), 1
        for _ in range(min(plies, rows * columns - 2)):
            legal = np.flatnonzero(fills < rows)
            j = int(rng.choice(legal))
            board[rows - 1 - fills[j], j] = turn
            fills[j] += 1
            if _has_line(board, turn, 4):
                break
            turn = -turn
        else:
            return board, fills, turn


def _gomoku_root(rng, rows, columns, stones):
    """`stones` stones placed alternately on random cells, none of which ended the game."""
    while True:
        board, turn = np.zeros((rows, columns), np.int8), 1
        for c in rng.permutation(rows * columns)[:stones]:
            board[c // columns, c % columns] = turn
            turn = -turn
        if not (_has_line(board, 1, 5) or _has_line(board, -1, 5)):
            return board, turn


def _tree(rng, nodes, edges):
    """One tree in the launcher's arrays as a search with full expansion leaves it: the most visited leaf is expanded
    next, visits spread over its children by their priors, a few leaves are ends of games."""
    child = np.full((nodes, edges), -1, np.int32)
    visits = np.zeros((nodes, edges), np.int32)
    quality = np.zeros((nodes, edges), np.float32)
    expanded = np.zeros(nodes, np.int32)
    node_visits = np.zeros(nodes, np.int64)
    node_visits[0] = 8 * nodes
    count, node = 1, 0
    while True:
        k = min(edges if edges < 16 else int(rng.integers(edges // 2, edges + 1)), nodes - count)
        if k < 1:
            break
        share = rng.gamma(0.5, size=k) + 1e-3
        mine = np.floor((node_visits[node] - 1) * share / share.sum()).astype(np.int64)
        child[node, :k] = np.arange(count, count + k)
        visits[node, :k] = np.minimum(mine, 1 << 20)
        quality[node, :k] = rng.uniform(-0.6, 0.6, size=k)
        expanded[node] = k
        node_visits[count:count + k] = mine
        count += k
        leaves = np.where(expanded[:count] == 0, node_visits[:count], -1)
        node = int(leaves.argmax())
    ends = (expanded[:count] == 0) & (rng.random(count) < 0.03)
    ends[0] = False
    expanded[:count][ends] = puct.NODE_EXPANDED_TERMINAL
    return child, visits, quality, expanded, count


def _forest(case, seed):
    trees, nodes, edges, warps, depth = (case[k] for k in ("trees", "nodes", "edges", "traversals", "depth"))
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    d = {}
    if case["shape"] == "deep":   # edge a of every node leads to node a + 1, everything expanded
        d["edge_child"] = torch.arange(1, edges + 1, dtype=torch.int32, device=DEVICE).expand(trees, nodes, edges).contiguous()
        d["edge_n"] = torch.ones((trees, nodes, edges), dtype=torch.int32, device=DEVICE)
        d["edge_w"] = torch.rand((trees, nodes, edges), generator=gen, device=DEVICE) - 0.5
        d["edge_prior"] = torch.rand((trees, nodes, edges), generator=gen, device=DEVICE) / edges
        d["node_expanded"] = torch.full((trees, nodes), edges, dtype=torch.int32, device=DEVICE)
        d["node_count"] = torch.full((trees,), nodes, dtype=torch.int32, device=DEVICE)
    else:
        shapes = [_tree(rng, nodes, edges) for _ in range(min(trees, 8))]
        which = torch.arange(trees, device=DEVICE) % len(shapes)

        def of_shapes(i):
            return torch.from_numpy(np.stack([s[i] for s in shapes])).to(DEVICE)[which]

        d["edge_child"], d["edge_n"], d["node_expanded"] = of_shapes(0), of_shapes(1), of_shapes(3)
        d["edge_w"] = d["edge_n"] * (of_shapes(2) + 0.2 * (torch.rand((trees, nodes, edges), generator=gen, device=DEVICE) - 0.5))
        prior = torch.rand((trees, nodes, edges), generator=gen, device=DEVICE).pow_(3) * (d["edge_child"] >= 0)
        d["edge_prior"] = prior / prior.sum(dim=2, keepdim=True).clamp_min(1e-6)
        d["node_count"] = torch.tensor([s[4] for s in shapes], dtype=torch.int32, device=DEVICE)[which]
    d["node_expand_inflight"] = torch.zeros((trees, nodes), dtype=torch.int32, device=DEVICE)
    if case["claims"] == "edge":
        d["edge_inflight"] = torch.zeros((trees, nodes, edges), dtype=torch.int32, device=DEVICE)
    else:
        d["node_inflight"] = torch.zeros((trees, nodes), dtype=torch.int32, device=DEVICE)
    d["out_selected"] = torch.zeros((trees, warps), dtype=torch.int32, device=DEVICE)
    d["out_path"] = torch.full((trees, warps, depth), -1, dtype=torch.int32, device=DEVICE)
    d["out_len"] = torch.zeros((trees, warps), dtype=torch.int32, device=DEVICE)
    # the leaves of a tree's batch are all valued alike, seen from the side to move level by level (which traversal takes
    # which path is theirs to race for)
    value = torch.rand((trees, 1, 1), generator=gen, device=DEVICE) * 2 - 1
    sign = 1.0 - 2.0 * (torch.arange(depth, device=DEVICE) % 2)
    values = (value * sign).expand(trees, warps, depth).contiguous()
    return d, values


def prepare(case, seed):
    state = dict(case=case)
    if case["kind"] == "select":
        state["trees"], state["values"] = _forest(case, seed)
        return state
    rng = np.random.default_rng(seed)
    rows, columns = case["rows"], case["columns"]
    if case["kind"] == "loop":
        state["root"] = _gomoku_root(rng, rows, columns, int(rng.integers(case["stones_low"], case["stones_high"] + 1)))
        state["engine"] = PUCTGomoku(board_shape=(rows, columns), trees=case["trees"], traversals=case["traversals"], max_nodes=case["nodes"],
                                     path_depth=case["depth"], cpuct=1.5, c_pw=case["c_pw"], dirichlet_alpha=0.3, seed=seed)
        return state
    state["engines"], state["roots"] = [], []
    for _ in range(case["searches"]):
        stones = int(rng.integers(case["stones_low"], case["stones_high"] + 1))
        if case["game"] == "c4":
            state["roots"].append(_c4_root(rng, rows, columns, stones))
            kw = dict(state_board_shape=(rows, columns), state_extra_info_memory=columns, state_max_actions=columns, game="c4",
                      action_index_to_name_function=C4.action_index_to_name)
        else:
            board, turn = _gomoku_root(rng, rows, columns, stones)
            state["roots"].append((board, None, turn))
            kw = dict(state_board_shape=(rows, columns), state_extra_info_memory=0, state_max_actions=rows * columns, game="gomoku")
        engine = MCTSNC(search_time_limit=np.inf, search_steps_limit=case["steps"], n_trees=case["trees"], n_playouts=case["playouts"],
                        variant=case["variant"], device_memory=case["memory"], ucb_c=2.0, seed=seed, verbose_info=False, **kw)
        engine.init_device_side_arrays()
        state["engines"].append(engine)
    return state


# ---- one pass ----------------------------------------------------------------------------------------------------------
def _answer(engine, table, values):
    """What a player's program reads after a move: the best action, the table of root actions, the trees' statistics."""
    info = engine.actions_info
    for a, e in info.items():
        if a != "best":
            table[a] = (e["n_root"], e["win_flag"], e["n"], e["n_wins"])
            values[a] = (e["q"], e["ucb"])
    trees = engine.performance_info["trees"]
    return (engine.best_action, engine.steps, trees["max_depth"], trees["max_size"]), (trees["mean_depth"], trees["mean_size"])


def run(state):
    case = state["case"]
    if case["kind"] == "select":
        d = state["trees"]
        if case["claims"] == "edge":
            puct.launch_select(d, cpuct=1.5, c_pw=0.0)
            puct.launch_edge_backup(d, None if case["shape"] == "deep" else state["values"])
        else:
            puct.launch_node_select(d, cpuct=1.5, c_pw=0.0, variant=case["rule"])
            puct.launch_node_backup(d, state["values"])
        out = {k: d[k] for k in ("edge_w", "edge_n", "node_expand_inflight", "edge_inflight", "node_inflight") if k in d}
        if case["traversals"] == 1:   # (with several, which of them takes which path is theirs to race for)
            out.update({k: d[k] for k in ("out_selected", "out_len", "out_path")})
        return out
    if case["kind"] == "loop":
        engine = state["engine"]
        engine.run(state["root"][0], state["root"][1], case["steps"])
        return {"best": engine.best_action, "root_n": engine.root_n, "root_q": engine.root_q, "selections": list(engine.selections.values()),
                "nodes": engine.performance_info["nodes_total"]}
    engines, roots = state["engines"], state["roots"]
    if len(engines) == 1:
        engines[0].run(*roots[0])
    else:
        boards, extras, turns = zip(*roots)
        run_batch(engines, boards, extras if extras[0] is not None else None, turns)
    actions = engines[0].state_max_actions
    table, values = np.full((len(engines), actions, 4), -1, np.int64), np.zeros((len(engines), actions, 2))
    answers = [_answer(e, t, v) for e, t, v in zip(engines, table, values)]
    return {"table": table, "values": values, "answers": np.array([a[0] for a in answers], np.int64), "trees": np.array([a[1] for a in answers])}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------
def work(case):
    """Bytes: inputs read and outputs written once.  `flops`: for searches the integer and floating operations of the
    playouts (about 40 a move: a generator step and its conversion, the move, the test for a line), for the PUCT paths 6 an
    edge scored."""
    if case["kind"] == "select":
        per_tree = 0
        fields = 5 if case["claims"] == "edge" else 4
        levels = case["depth"] if case["shape"] == "deep" else max(2.0, math.log(case["nodes"]) / math.log(4.0))
        # (traversals of one tree share the upper levels: a row is read once by whoever needs it first)
        rows = levels if case["shape"] == "deep" else 1 + (levels - 1) * (1 + 0.3 * (case["traversals"] - 1))
        rows = min(rows, case["nodes"])
        per_tree += rows * (fields * 4 * case["edges"] + 8) + case["traversals"] * (levels * 20 + 8)
        return {"bytes": case["trees"] * per_tree, "flops": case["trees"] * case["traversals"] * levels * case["edges"] * 6}
    cells = case["rows"] * case["columns"]
    if case["kind"] == "loop":
        leaves = case["trees"] * case["traversals"] * case["steps"] * (1.0 if case["c_pw"] >= case["traversals"] else 0.25)
        return {"bytes": leaves * (160 + 17 * cells), "flops": leaves * 60 * cells}
    trees = case["trees"] * case["searches"]
    acp = case["variant"].startswith("acp")
    actions = case["columns"] if case["game"] == "c4" else cells
    streams = trees * case["playouts"] * (actions if acp else 1)
    # (a Connect 4 step often ends at a decided position and plays nothing)
    played = (0.35 * actions if case["game"] == "c4" else 0.95 * actions) if acp else (0.7 if case["game"] == "c4" else 1.0)
    plies = 8 if case["game"] == "c4" else 0.45 * cells
    node = 32 + cells / 4
    return {"bytes": 32 * streams + trees * case["steps"] * (0.35 * actions if case["game"] == "c4" else 0.95 * actions) * node,
            "flops": trees * case["steps"] * played * case["playouts"] * plies * 40}


def tolerance(case):
    if case["kind"] == "select" and case["traversals"] > 1:
        # the traversals of a tree race for their claims: a few of the visits of one selection land on other edges
        return {"rel": 1e-2, "max": 0.99, "differ": 0.01}
    return "exact"
