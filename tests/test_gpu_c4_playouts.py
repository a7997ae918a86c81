"""Connect 4 playouts at the edges of their two board layouts, engine against oracle, every array bit for bit (two searches
in a row): boards whose columns each fit one of the two words and whose fours start in the lower one (4 x 4 to 7 x 7, a lower
word of four to six columns, with and without free bits below them), the first ones that miss either condition, by teams, by
one workgroup per tree, by teams with playout pools and by teams that split playouts over wavefronts; searches long enough to
meet draws rounded up to 1.0f; and playouts split over wavefronts, in each number of workgroups to a column, on full and nearly
decided boards, and where the split form is not the one taken by itself."""
import numpy as np
import pytest

from helpers import compare_with_oracle, make_engine, random_c4_root
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

FORMS = dict(teams=dict(solo_trees=0, team_pool=0, split=0), solo=dict(solo_trees=1), pools=dict(solo_trees=0, team_pool=1), split=dict(solo_trees=0, team_pool=0, split=1))
BOARDS = [(4, 4), (6, 4), (5, 6), (4, 7), (5, 8), (6, 6), (7, 7), (7, 4), (8, 6), (6, 8), (4, 8)]
LONG = [  # rows, columns, plies, variant, seed, steps: the oracle meets at least one such draw in each
    (6, 7, 0, "acp_prodigal", 0, 150), (5, 6, 0, "acp_prodigal", 0, 150), (7, 8, 0, "acp_prodigal", 0, 150),
    (6, 7, 2, "ocp_thrifty", 5, 600), (5, 6, 2, "ocp_thrifty", 5, 600),
]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n", BOARDS)
def test_playouts_on_both_board_layouts(m, n, form):
    params = dict(n_trees=2, n_playouts=64, variant="acp_prodigal", device_memory=0.1, ucb_c=2.0, seed=3)
    e = make_engine(params, board_shape=(m, n), extra=n, actions=n, options=FORMS[form])
    o = Oracle("c4", (m, n), n, n, 2, 64, "acp_prodigal", ucb_c=2.0, seed=3, device_memory=0.1, threads=8)
    rng = np.random.default_rng(10 * m + n)
    for plies in (0, m * n // 2):
        board, fills, turn = random_c4_root(rng, plies, m, n)
        compare_with_oracle(e, o, board, fills, turn, steps=120)


@pytest.mark.parametrize("m,n,plies,variant,seed,steps", LONG)
def test_draws_rounded_up_are_replayed(m, n, plies, variant, seed, steps):
    params = dict(n_trees=4, n_playouts=512, variant=variant, device_memory=0.3, ucb_c=2.0, seed=seed)
    for options in [FORMS[form] for form in ("teams", "solo", "pools")] if variant.startswith("acp") else (None,):   # (512 playouts are never split)
        e = make_engine(params, board_shape=(m, n), extra=n, actions=n, options=options)
        o = Oracle("c4", (m, n), n, n, 4, 512, variant, ucb_c=2.0, seed=seed, device_memory=0.3, threads=8)
        compare_with_oracle(e, o, *random_c4_root(np.random.default_rng(seed), plies, m, n), steps=steps)
        assert o.u1_events > 0


SPLIT = [  # rows, columns, variant, trees, playouts, plies, steps, memory (GiB), seed
    (6, 7, "acp_prodigal", 4, 256, 0, 150, 0.3, 5), (7, 8, "acp_thrifty", 4, 256, 0, 150, 0.3, 5), (6, 7, "ocp_thrifty", 8, 64, 0, 900, 0.3, 5),
    (8, 6, "ocp_prodigal", 9, 32, 1, 400, 0.3, 1), (4, 4, "ocp_thrifty", 1, 1, 9, 200, 0.1, 2), (6, 7, "acp_thrifty", 8, 128, 5, 200, 0.3, 3),
    (4, 4, "acp_prodigal", 3, 64, 0, 700, 0.1, 4), (5, 8, "acp_prodigal", 2, 128, 22, 400, 0.1, 6), (6, 7, "acp_prodigal", 2, 256, 26, 1500, 0.1, 7),
    (6, 7, "acp_thrifty", 4, 256, 26, 900, 0.001, 8), (7, 4, "acp_prodigal", 8, 2, 3, 300, 0.1, 9),
    (6, 7, "acp_prodigal", 2, 128, 8, 400, 0.1, 22),
]


@pytest.mark.parametrize("m,n,variant,trees,playouts,plies,steps,memory,seed", SPLIT)
def test_playouts_split_over_wavefronts(m, n, variant, trees, playouts, plies, steps, memory, seed):
    """The first three meet a draw rounded up to 1.0f; those with many stones end at terminal nodes for long stretches, in which
    teams stop exchanging results; the one with little memory fills its pool."""
    params = dict(n_trees=trees, n_playouts=playouts, variant=variant, device_memory=memory, ucb_c=2.0, seed=seed)
    e = make_engine(params, board_shape=(m, n), extra=n, actions=n)
    o = Oracle("c4", (m, n), n, n, trees, playouts, variant, ucb_c=2.0, seed=seed, device_memory=memory, threads=8)
    for extra in (0, 1):
        compare_with_oracle(e, o, *random_c4_root(np.random.default_rng(seed + extra), plies, m, n), steps=steps)
    if seed == 5:
        assert o.u1_events > 0


@pytest.mark.parametrize("split", [0, 1])
@pytest.mark.parametrize("m,n,variant,trees,playouts,plies,steps", [
    (6, 7, "acp_prodigal", 4, 256, 0, 150), (6, 7, "acp_thrifty", 2, 128, 30, 600), (5, 6, "acp_prodigal", 3, 64, 20, 500), (6, 7, "ocp_thrifty", 8, 64, 4, 400),
    (7, 8, "ocp_prodigal", 2, 16, 0, 300),
])
def test_both_forms_of_small_searches(m, n, variant, trees, playouts, plies, steps, split):
    """Searches that fit the split form, with it and without (nearly full boards of all-children variants: without is the default)."""
    params = dict(n_trees=trees, n_playouts=playouts, variant=variant, device_memory=0.2, ucb_c=2.0, seed=11)
    e = make_engine(params, board_shape=(m, n), extra=n, actions=n, options=dict(split=split))
    o = Oracle("c4", (m, n), n, n, trees, playouts, variant, ucb_c=2.0, seed=11, device_memory=0.2, threads=8)
    compare_with_oracle(e, o, *random_c4_root(np.random.default_rng(plies), plies, m, n), steps=steps)
