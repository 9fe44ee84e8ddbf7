"""Distance fields of maps whose rows do not fit one 64-bit word per lane
(more than 4,096 cells): every way the row search lays a map over lanes and
wavefronts, at its edges, against the C oracle.

Each shape has four envs: i.i.d. obstacles, no obstacle at all (the largest
levels of ordinary maps), a maze, and a serpentine corridor whose levels use
every level bit a map of that size can (its level planes past the register
ones).  Goals lie in the corners, at the corridor's ends, on obstacles and at
random, agents on free cells, walls and cells without a way to their goal.
Distances, tokens, greedy masks and diagnostics are whole numbers: equal.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SHAPES = [
    # four rows per lane, the last lanes' rows past the map
    (130, 32), (256, 32), (129, 64), (256, 64),
    # two rows per lane up to 128 rows, split beyond (two and three wavefronts)
    (65, 64), (128, 64), (65, 96), (128, 96), (129, 96), (240, 96), (241, 96), (127, 128), (128, 128), (129, 128),
    (240, 128), (256, 128),
    # one row per lane up to 64 rows, split beyond (two to five wavefronts)
    (43, 96), (33, 128), (64, 128), (26, 160), (64, 160), (65, 160), (112, 160), (113, 192), (64, 192), (160, 224),
    (64, 224), (17, 256), (64, 256), (161, 256), (208, 256), (209, 256), (256, 256),
]


def serpentine(W, H):
    g = np.ones((W, H), np.uint8)
    g[::2, :] = 0
    for i, x in enumerate(range(1, W - 1, 2)):
        g[x, H - 1 if i % 2 == 0 else 0] = 0
    return g


def four_maps(W, H, seed):
    from iclr_2027_jointoom_amd.synthetic import iid_grid, maze_grid

    rng = np.random.default_rng(seed)
    return np.stack([(rng.random((W, H)) < 0.2).astype(np.uint8), np.zeros((W, H), np.uint8), maze_grid(rng, W, H),
                     serpentine(W, H)])


def pick(rng, grid, n, corners):
    """n cells: the free cells nearest the corners, one obstacle (if any), the rest free."""
    W, H = grid.shape
    free = np.argwhere(grid == 0)
    out = [free[np.abs(free - c).sum(1).argmin()] for c in ([0, 0], [W - 1, H - 1], [0, H - 1])[:corners]]
    walls = np.argwhere(grid != 0)
    if len(walls):
        out.append(walls[rng.integers(len(walls))])
    out += list(free[rng.integers(len(free), size=n - len(out))])
    return np.array(out)


def build_and_compare(oracle, grids, pos, goals, rounds=((),)):
    """Builds from state; each round replaces the goals of the agents it names; the last state's fields too."""
    from iclr_2027_jointoom_amd import profile

    E, W, H = grids.shape
    A = pos.shape[1]
    builder = profile(W, H).MapfGPTObservationBuilder(torch.from_numpy(grids.astype(np.int32)).cuda(), A)
    ob = oracle.OracleMapfGPT(grids, A)
    goals = goals.astype(np.int16).copy()
    pos = pos.astype(np.int16)
    for change in rounds:
        for (e, a), cell in change:
            goals[e, a] = cell
        st = [np.ascontiguousarray(v) for v in (pos[..., 0], pos[..., 1], goals[..., 0], goals[..., 1])]
        builder.build_tokens_from_state(*(torch.from_numpy(v).cuda() for v in st))
        ob.build_state(*st)
        torch.cuda.synchronize()
        assert np.array_equal(builder.cost_to_go.cpu().numpy().view(np.uint16), ob.cost_to_go)
        assert np.array_equal(builder.tokens.cpu().numpy(), ob.tokens)
        assert builder.diagnostics.cpu().tolist() == ob.diagnostics.tolist()
    return ob


@pytest.mark.parametrize("W,H", SHAPES)
def test_fields_of_every_layout(oracle, W, H):
    grids = four_maps(W, H, W * 1000 + H)
    rng = np.random.default_rng(W + H)
    A = 7
    goals = np.stack([pick(rng, g, A, 3) for g in grids])
    pos = np.stack([pick(rng, g, A, 1) for g in grids])
    # one goal of each env changes after the first build, the others' fields are kept
    free = [np.argwhere(g == 0) for g in grids]
    change = [((e, e + 2), free[e][rng.integers(len(free[e]))]) for e in range(len(grids))]
    build_and_compare(oracle, grids, pos, goals, ((), change))


@pytest.mark.parametrize("W,H,E,A", [(128, 128, 40, 100), (256, 256, 7, 150), (100, 96, 3, 1100)])
def test_more_fields_than_workgroups(oracle, W, H, E, A):
    """Every goal new, several fields per wavefront and workgroup; then a few."""
    rng = np.random.default_rng(W * H + A)
    grids = (rng.random((E, W, H)) < 0.15).astype(np.uint8)
    free = [np.argwhere(g == 0) for g in grids]
    pos = np.stack([f[rng.choice(len(f), A, replace=False)] for f in free])
    goals = np.stack([f[rng.choice(len(f), A, replace=False)] for f in free])
    change = [((int(e), int(a)), free[int(e)][0]) for e, a in zip(rng.integers(0, E, 9), rng.integers(0, A, 9))]
    build_and_compare(oracle, grids, pos, goals, ((), change))


def level_of_many_cells():
    """A 256x256 map whose last level holds more than 4,096 cells: an H-tree
    of corridors (4,096 leaves, all as far from the root) with further cells
    hung on the cells just before that level."""
    n = 256
    free = np.zeros((n, n), bool)

    def tree(x, y, half, across):
        if half < 1:
            return
        if across:
            free[max(0, x - half):x + half + 1, y] = True
            tree(x - half, y, half, False)
            tree(x + half, y, half, False)
        else:
            free[x, max(0, y - half):y + half + 1] = True
            rest = 0 if half == 2 else half // 2
            tree(x, y - half, rest, True)
            tree(x, y + half, rest, True)

    tree(n // 2, n // 2, n // 4, True)
    return free


def test_level_past_the_frontier_limit(oracle):
    """diagnostics[0] counts the cells of a level past 4,096 (the whole search
    split over five wavefronts)."""
    free = level_of_many_cells()
    root = (128, 128)
    field = oracle.bfs_u16((~free).astype(np.uint8), root)[0]
    last = int(field[free].max())
    hung = 0
    for x, y in np.argwhere(~free):
        near = [(x + dx, y + dy) for dx, dy in ((-1, 0), (1, 0), (0, -1), (0, 1))
                if 0 <= x + dx < 256 and 0 <= y + dy < 256 and free[x + dx, y + dy]]
        if len(near) == 1 and field[near[0]] == last - 1:
            free[x, y] = True
            field[x, y] = last
            hung += 1
    assert hung > 100
    grids = (~free).astype(np.uint8)[None]
    cells = np.argwhere(free)
    goals = np.array([root, cells[0], cells[-1], root])[None]
    pos = cells[[5, 50, 500, 5000]][None]
    ob = build_and_compare(oracle, grids, pos, goals)
    assert ob.diagnostics[0] >= 2 * hung
