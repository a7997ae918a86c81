"""Gomoku playouts at the edges of their formats, engine against oracle, every array bit for bit (two searches in a row):
the boards on either side of the narrow format's limits (rows of 15 cells, on their side or not; 16 x 16 is the first wide
one), the widest ones (22 rows, 32 columns), playout counts on either side of what a 16-byte store, a wavefront and a round
of the workgroup hold, and children whose playouts are cut into several rounds or share one."""
import numpy as np
import pytest

from helpers import compare_with_oracle, make_engine, random_gomoku_root
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

CASES = [  # rows, columns, stones, variant, trees, playouts, steps
    (16, 15, 40, "ocp_thrifty", 2, 64, 20), (15, 16, 40, "acp_prodigal", 1, 32, 4), (16, 16, 3, "ocp_prodigal", 1, 128, 12),
    (16, 16, 90, "acp_thrifty", 2, 64, 3), (5, 5, 0, "acp_prodigal", 3, 512, 30), (5, 32, 20, "ocp_thrifty", 1, 256, 12),
    (22, 23, 100, "ocp_prodigal", 1, 128, 8), (32, 16, 60, "acp_prodigal", 1, 16, 2), (15, 15, 12, "ocp_thrifty", 2, 512, 12),
    (15, 15, 150, "acp_thrifty", 3, 1, 12), (13, 9, 50, "acp_prodigal", 4, 2, 12), (12, 16, 30, "ocp_thrifty", 2, 8, 40),
    (19, 19, 150, "acp_prodigal", 2, 1, 4), (19, 19, 30, "ocp_thrifty", 1, 2, 40), (9, 9, 60, "acp_prodigal", 300, 16, 4),
    (9, 9, 20, "ocp_prodigal", 300, 128, 6),
]


@pytest.mark.parametrize("m,n,stones,variant,trees,playouts,steps", CASES)
def test_playouts_at_the_edges_of_their_formats(m, n, stones, variant, trees, playouts, steps):
    rng = np.random.default_rng(m * 1000 + n * 10 + playouts)
    params = dict(n_trees=trees, n_playouts=playouts, variant=variant, device_memory=0.3, ucb_c=2.0, seed=int(rng.integers(1000)))
    e = make_engine(params, board_shape=(m, n), extra=0, actions=m * n, game="gomoku")
    o = Oracle("gomoku", (m, n), 0, m * n, trees, playouts, variant, ucb_c=2.0, seed=params["seed"], device_memory=0.3, threads=8)
    for _ in range(2):
        board, turn = random_gomoku_root(rng, m, n, stones)
        compare_with_oracle(e, o, board, None, turn, steps)


# boards around the fewest cells for which ends are looked for up to a limit first (169 and 170), the largest ones whose marked
# times fit a byte, roots that leave few plies to the limit, draws on either side of a chunk and of what is worth leaving, more
# groups of 64 playouts than boards of times, and enough playouts that many outlast the limit
LONG_GAMES = [
    (10, 17, 0, "acp_prodigal", 2, 64, 4), (13, 13, 0, "ocp_thrifty", 4, 256, 12), (13, 13, 30, "acp_thrifty", 3, 64, 6), (13, 14, 60, "acp_prodigal", 2, 128, 4),
    (15, 15, 0, "ocp_prodigal", 4, 256, 16), (15, 15, 90, "acp_prodigal", 2, 64, 6), (15, 15, 14, "acp_thrifty", 2, 32, 8), (16, 15, 0, "acp_thrifty", 1, 64, 5),
    (15, 16, 1, "ocp_thrifty", 3, 128, 12), (16, 16, 0, "acp_prodigal", 1, 64, 4), (19, 19, 100, "acp_prodigal", 1, 32, 3), (19, 19, 2, "ocp_thrifty", 4, 128, 12),
    (22, 23, 0, "ocp_thrifty", 2, 256, 6), (16, 14, 0, "ocp_prodigal", 300, 128, 4), (15, 15, 9, "ocp_thrifty", 2, 512, 12), (32, 16, 40, "ocp_prodigal", 1, 256, 6),
] + [(15, 14, stones, "ocp_thrifty", 3, 256, 5) for stones in (20, 27, 28, 100, 130, 140)] + [(17, 17, stones, "ocp_prodigal", 3, 128, 5) for stones in (0, 7, 150, 200)]


@pytest.mark.parametrize("m,n,stones,variant,trees,playouts,steps", LONG_GAMES)
def test_games_that_outlast_the_first_look_for_their_end(m, n, stones, variant, trees, playouts, steps):
    test_playouts_at_the_edges_of_their_formats(m, n, stones, variant, trees, playouts, steps)
