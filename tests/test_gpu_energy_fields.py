"""uint8 energy fields (255 - distance, 0 past 254) from the row search, in
every way it lays a map over lanes and wavefronts, against the C oracle: i.i.d.
maps, maps without an obstacle, mazes and a serpentine (distances past the cap
at every phase of a batch of 16 levels), goals in corners, at random, on
obstacles and off the map, rows of envs and agents that do not exist."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 32), (64, 32), (65, 32), (129, 32), (256, 32), (33, 64), (64, 64), (65, 64), (129, 64), (256, 64),
    (64, 96), (128, 96), (129, 96), (241, 96), (128, 128), (129, 128), (256, 128), (64, 160), (65, 160), (160, 192),
    (113, 224), (16, 256), (64, 256), (209, 256), (256, 256),
]


def serpentine(W, H):
    g = np.ones((W, H), np.uint8)
    g[::2, :] = 0
    for i, x in enumerate(range(1, W - 1, 2)):
        g[x, H - 1 if i % 2 == 0 else 0] = 0
    return g


def maps(W, H, seed):
    from iclr_2027_jointoom_amd.synthetic import maze_grid

    rng = np.random.default_rng(seed)
    third = maze_grid(rng, W, H) if W >= 8 else (rng.random((W, H)) < 0.4).astype(np.uint8)
    return np.stack([(rng.random((W, H)) < 0.2).astype(np.uint8), np.zeros((W, H), np.uint8), third, serpentine(W, H)])


def state_rows(rng, grids, A):
    E, W, H = grids.shape
    rows = np.zeros((E, A, 8), np.int16)
    rows[..., 0] = np.arange(E)[:, None]
    rows[..., 1] = np.arange(A)[None]
    rows[..., 4] = rng.integers(0, W, (E, A))  # free or not
    rows[..., 5] = rng.integers(0, H, (E, A))
    rows[:, 0, 4:6] = 0
    rows[:, 1, 4:6] = W - 1, H - 1
    rows[..., 7] = 1
    return rows


@pytest.mark.parametrize("W,H", SHAPES)
def test_energy_of_every_layout(oracle, W, H):
    from iclr_2027_jointoom_amd import profile

    rng = np.random.default_rng(W * 7 + H)
    grids, A = maps(W, H, W + H), 9
    rows = state_rows(rng, grids, A)
    rows[2, 5, 4] = W  # off the map
    rows[1, 6, 5] = -1
    rows[3, 7, 0] = 4  # no such env
    rows[0, 8, 1] = A  # no such agent
    flat = rows.reshape(-1, 8)
    sim = profile(W, H).StatelessGridWorldSimulator(torch.from_numpy(grids.astype(np.int32)).cuda(), A, 3)
    m = oracle.OracleMagat(grids, A)
    sim.update_energy_maps(torch.from_numpy(flat).cuda(), len(flat))
    m.update_energy(flat.view(np.uint16), len(flat))
    torch.cuda.synchronize()
    assert np.array_equal(sim.energy_maps.cpu().numpy(), m.energy)


@pytest.mark.parametrize("W,H,E,A", [(64, 64, 40, 130), (128, 128, 30, 200), (256, 256, 3, 400)])
def test_many_fields_then_the_flagged_ones(oracle, W, H, E, A):
    """More jobs than resident wavefronts or workgroups; then, through the
    simulator, every field (its first step) and only those whose goal changed,
    the others' left as they are."""
    from iclr_2027_jointoom_amd import profile

    rng = np.random.default_rng(W + E)
    grids = (rng.random((E, W, H)) < 0.2).astype(np.uint8)
    free = [np.argwhere(g == 0) for g in grids]
    pos = np.stack([f[rng.choice(len(f), A, replace=False)] for f in free]).astype(np.int16)
    goals = np.stack([f[rng.choice(len(f), A, replace=False)] for f in free]).astype(np.int16)
    g = torch.from_numpy(grids.astype(np.int32)).cuda()
    rows = state_rows(rng, grids, A)
    rows[..., 4:6] = goals
    flat = rows.reshape(-1, 8)
    want = oracle.energy_maps(grids, flat.view(np.uint16), len(flat), A)
    stateless = profile(W, H).StatelessGridWorldSimulator(g, A, 3)
    stateless.update_energy_maps(torch.from_numpy(flat).cuda(), len(flat))
    assert np.array_equal(stateless.energy_maps.cpu().numpy(), want)
    sim = profile(W, H).GridWorldSimulator(g, A, 0, E * W * H, 1, "standard_mapf", 64)
    sim.load_state(torch.from_numpy(pos).cuda(), torch.from_numpy(goals).cuda(),
                   torch.zeros((E, A), dtype=torch.uint8, device="cuda"), torch.zeros(E, dtype=torch.int32, device="cuda"))
    sim.current_step = 1
    sim.update_derived_state()
    assert np.array_equal(sim.energy_maps.cpu().numpy(), want)
    flags = np.zeros((E, A), np.uint8)
    for e, a in zip(rng.integers(0, E, 11), rng.integers(0, A, 11)):
        flags[e, a] = 1
        goals[e, a] = free[e][0]
        rows[e, a, 4:6] = free[e][0]
    sim.current_step = 2
    sim.goal_changed_flags.copy_(torch.from_numpy(flags).cuda())
    sim.goal_x.copy_(torch.from_numpy(goals[..., 0].copy()).cuda())
    sim.goal_y.copy_(torch.from_numpy(goals[..., 1].copy()).cuda())
    sim.update_derived_state()
    torch.cuda.synchronize()
    assert np.array_equal(sim.energy_maps.cpu().numpy(), oracle.energy_maps(grids, flat.view(np.uint16), len(flat), A))
    packed = sim.changed_state_packed.cpu().numpy()
    e, a = np.nonzero(flags)
    assert int(sim.goal_changed_count.item()) == len(e)
    assert np.array_equal(packed[: len(e), :2], np.stack([e, a], 1)) and not packed[len(e):].any()


@pytest.mark.parametrize("W,H", [(16, 256), (13, 256), (1, 256), (18, 224), (64, 64), (64, 32)])
def test_refresh_of_changed_goals_in_one_launch(oracle, W, H):
    """Maps of at most 4,096 cells and 64 rows: scan, packed rows and the
    changed goals' fields (of distances past the cap) in a single launch."""
    from iclr_2027_jointoom_amd import profile
    from launches import launches

    rng = np.random.default_rng(W * 3 + H)
    grids, A = maps(W, H, W + H), 40
    E = len(grids)
    rows = state_rows(rng, grids, A)
    goals = np.ascontiguousarray(rows[..., 4:6])
    sim = profile(W, H).GridWorldSimulator(torch.from_numpy(grids.astype(np.int32)).cuda(), A, 0, E * W * H, 1,
                                           "standard_mapf", 64)
    sim.load_state(torch.from_numpy(goals).cuda(), torch.from_numpy(goals).cuda(),
                   torch.zeros((E, A), dtype=torch.uint8, device="cuda"), torch.zeros(E, dtype=torch.int32, device="cuda"))
    flags = (rng.random((E, A)) < 0.6).astype(np.uint8)
    sim.current_step = 2
    sim.goal_changed_flags.copy_(torch.from_numpy(flags).cuda())
    sim.energy_maps.fill_(7)
    sim.update_derived_state()
    torch.cuda.synchronize()
    flat = rows.reshape(-1, 8)
    want = oracle.energy_maps(grids, flat.view(np.uint16), len(flat), A).reshape(E, A, -1)
    got = sim.energy_maps.cpu().numpy().reshape(E, A, -1)
    assert np.array_equal(got[flags == 1], want[flags == 1]) and (got[flags == 0] == 7).all()
    assert [k.name for k in launches(sim.update_derived_state) if "refresh_kernel" not in k.name] == []
