"""Distance fields of maps of at most 64 x 64 cells, whose searches hold a
row's even and odd columns apart: every parity of start and row, goals without
a free neighbour, in the corners and on obstacles, corridors of the most
levels such a map can have, rows of 32 columns (half a word per colour) and of
64, fewer rows than lanes; against the C oracle.  Whole numbers: equal.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_large_fields import build_and_compare, four_maps, pick  # noqa: E402


@pytest.mark.parametrize("W,H", [(64, 64), (63, 64), (33, 64), (8, 64), (64, 32), (61, 32), (9, 32)])
def test_fields_of_both_colours(oracle, W, H):
    rng = np.random.default_rng(W * 100 + H)
    grids = four_maps(W, H, W * 1000 + H)
    alone = np.ones((1, W, H), np.uint8)  # free cells without a free neighbour, one component of two cells
    for x, y in ((0, 0), (1, 1), (2, 0), (W - 1, H - 1), (W - 2, H - 2), (4, 4), (4, 5), (6, H - 1), (5, 30)):
        alone[0, x, y] = 0
    grids = np.concatenate([grids, alone])
    A = 9
    goals = np.stack([pick(rng, g, A, 3) for g in grids])
    pos = np.stack([pick(rng, g, A, 1) for g in grids])
    goals[4], pos[4] = np.argwhere(grids[4] == 0), np.argwhere(grids[4] == 0)[rng.permutation(A)]
    # the goals of an open map: both parities of row and column
    goals[1, 3:7] = [(1, 0), (0, 1), (W - 2, H - 1), (3, 31)]
    change = [((e, 2 + e), np.argwhere(grids[e] == 0)[-1 - e]) for e in range(len(grids))]
    build_and_compare(oracle, grids, pos, goals, ((), change))
