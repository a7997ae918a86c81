"""Gomoku PUCT loop: the ways a group of traversals decides on a node, GPU against host oracle, array for array: no edge yet
(tickets, and too few of them), one edge, up to a row of 16, up to 64, more; every score equal (no exploration: the rotated
order decides), scores beyond what a row of lanes takes, no widening, and numbers of traversals that leave an evaluator two,
three or four nodes at a time."""
import numpy as np
import pytest

from helpers import random_gomoku_root
from oracle import puct_oracle as po
from test_gpu_puct_gomoku import assert_same_trees, read_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,traversals,cpuct,c_pw,steps", [
    ((15, 15), 16, 0.0, 16.0, 120), ((15, 15), 16, 0.0, 1.0, 200), ((9, 9), 12, 1e31, 4.0, 150), ((15, 15), 9, 1e36, 16.0, 100),
    ((15, 15), 16, 1.5, 0.0, 150), ((12, 12), 3, 1.5, 0.3, 400), ((15, 15), 4, 1e-3, 40.0, 250), ((8, 8), 2, 3.0, 5.0, 400),
    ((6, 6), 12, 0.5, 7.5, 250), ((16, 16), 16, 50.0, 40.0, 120)])
def test_every_way_of_deciding_equals_the_oracle(shape, traversals, cpuct, c_pw, steps):
    from mcts_numba_cuda_amd.puct_gomoku import PUCTGomoku
    board, turn = random_gomoku_root(np.random.default_rng(traversals), shape[0], shape[1], 4)
    kw = dict(trees=2, traversals=traversals, max_nodes=8192, path_depth=64, cpuct=cpuct, c_pw=c_pw, dirichlet_alpha=0.3, seed=5)
    want = po.gomoku_search(board, turn, steps, **kw)
    for fused, evaluators in ((True, 3), (True, 1), (True, 0), (False, 0)):
        with PUCTGomoku(board_shape=shape, evaluators=evaluators, **kw) as e:
            e.run(board, turn, steps, fused=fused)
            assert_same_trees(read_all(e), want)


@pytest.mark.parametrize("shape,traversals,c_pw,alpha_pw,cpuct,steps", [
    ((15, 15), 5, 1150.0, -2.0, 1.5, 60), ((9, 9), 4, 300.3, -1.5, 0.3, 80), ((15, 15), 16, 9001.0, -2.0, 1.5, 40), ((12, 12), 7, 37.3, -0.5, 5.0, 100),
    ((15, 15), 6, 1150.0, -2.0, 0.0, 60), ((15, 15), 8, 0.7, 0.9, 1.5, 80), ((9, 9), 6, 2.3, 0.0, 1.5, 80)])
def test_widening_limits_that_fall_with_the_visits_equal_the_oracle(shape, traversals, c_pw, alpha_pw, cpuct, steps):
    """A negative alpha_pw: of the traversals that decide on a node, those before the first claim see the largest widening limit, and get the tickets
    that it leaves.  (c_pw keeps the limits off whole numbers, where a last bit of powf would decide.)"""
    from mcts_numba_cuda_amd.puct_gomoku import PUCTGomoku
    board, turn = random_gomoku_root(np.random.default_rng(traversals), shape[0], shape[1], 4)
    kw = dict(trees=4, traversals=traversals, max_nodes=4096, path_depth=64, cpuct=cpuct, c_pw=c_pw, alpha_pw=alpha_pw, dirichlet_alpha=0.3, seed=5)
    want = po.gomoku_search(board, turn, steps, **kw)
    for fused, evaluators in ((True, 3), (False, 0)):
        with PUCTGomoku(board_shape=shape, evaluators=evaluators, **kw) as e:
            e.run(board, turn, steps, fused=fused)
            assert_same_trees(read_all(e), want)
