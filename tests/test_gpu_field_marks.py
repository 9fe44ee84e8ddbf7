"""Whether a field of a map of more than 4,096 cells carries greedy marks
(levels of at most 4,080) or plain distances belongs to the field itself:
every reader has to tell the two apart whatever other buffers hold.  Against
the CPU oracle, bit-exact, on maps whose fields are of both kinds."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N = 128


def mixed_maps():
    """A serpentine corridor (every field plain), an open map (every field
    marked), and both halves in one map, a wall between them."""
    snake = np.ones((N, N), np.uint8)
    snake[::2, :] = 0
    for i, x in enumerate(range(1, N - 1, 2)):
        snake[x, N - 1 if i % 2 == 0 else 0] = 0
    both = snake.copy()
    both[102:, :] = 0
    both[101, :] = 1
    return np.stack([snake, np.zeros((N, N), np.uint8), both])


def next_to_goals(grids, A, seed):
    """Goals on distinct free cells (of the third map every other one in its
    corridor), each agent on a free cell beside its goal, and the action that
    reaches it."""
    rng = np.random.default_rng(seed)
    E = len(grids)
    pos, goal = np.zeros((E, A, 2), np.int16), np.zeros((E, A, 2), np.int16)
    acts = np.zeros((E, A), np.uint8)
    for e, g in enumerate(grids):
        cells = [tuple(int(v) for v in c) for c in rng.permutation(np.argwhere(g == 0))]
        if e == 2:
            low, high = [c for c in cells if c[0] < 101], [c for c in cells if c[0] > 101]
            cells = [c for pair in zip(low, high) for c in pair]
        taken, a = set(), 0
        for x, y in cells:
            if a == A:
                break
            for act, (dx, dy) in enumerate(((-1, 0), (1, 0), (0, -1), (0, 1)), 1):
                sx, sy = x - dx, y - dy
                free = 0 <= sx < N and 0 <= sy < N and not g[sx, sy]
                if free and not taken & {(x, y), (sx, sy)}:
                    taken |= {(x, y), (sx, sy)}
                    goal[e, a], pos[e, a], acts[e, a] = (x, y), (sx, sy), act
                    a += 1
                    break
    return pos, goal, acts


def test_builds_do_not_read_an_old_agent_info(oracle):
    """agent_info is scratch: a caller may share it between builders or
    overwrite it between builds."""
    from iclr_2027_jointoom_amd import profile

    A = 20
    grids = mixed_maps()
    pos, goal, _ = next_to_goals(grids, A, 3)
    builder = profile(N, N).MapfGPTObservationBuilder(torch.from_numpy(grids.astype(np.int32)).cuda(), A)
    ob = oracle.OracleMapfGPT(grids, A)
    for word in (0, 0x80, 0xFFFFFFFF, 0x1234567F):
        builder._agent_info.fill_(word - (1 << 32) if word >> 31 else word)
        st = [np.ascontiguousarray(v) for v in (pos[..., 0], pos[..., 1], goal[..., 0], goal[..., 1])]
        builder.build_tokens_from_state(*(torch.from_numpy(v).cuda() for v in st))
        ob.build_state(*st)
        builder._agent_info.fill_(word - (1 << 32) if word >> 31 else word)
        assert np.array_equal(builder.tokens.cpu().numpy(), ob.tokens), hex(word)
        assert np.array_equal(builder.cost_to_go.cpu().numpy().view(np.uint16), ob.cost_to_go), hex(word)
        assert builder.diagnostics.cpu().tolist() == ob.diagnostics.tolist(), hex(word)
        # fields that turn from plain to marked and back, the others kept
        goal[2, :6] = np.roll(goal[2, :6], 1, 0)


@pytest.mark.parametrize("with_info", [True, False])
def test_costtracer_on_plain_and_marked_fields(oracle, with_info):
    """The CostTracer calls read the fields of the builder they are given and
    nothing else of it: also without an agent_info."""
    from iclr_2027_jointoom_amd import profile
    from iclr_2027_jointoom_amd.grid_world import _stream
    from oracle.costtracer import OracleCostTracer

    A, steps, horizon = 24, 6, 16
    grids = mixed_maps()
    E = len(grids)
    pos, goal, acts = next_to_goals(grids, A, 11)
    targets = np.stack([np.roll(goal, k + 1, axis=1) for k in range(horizon + 1)], axis=2).astype(np.int16)
    ext = profile(N, N)
    g = torch.from_numpy(grids.astype(np.int32)).cuda()
    sim = ext.GridWorldSimulator(g, A, 0, E * N * N, 3, "costtracer", horizon)
    builder = ext.MapfGPTObservationBuilder(g, A)
    dev = "cuda"
    sim.load_state(torch.from_numpy(pos).to(dev), torch.from_numpy(goal).to(dev),
                   torch.zeros((E, A), dtype=torch.uint8, device=dev), torch.zeros(E, dtype=torch.int32, device=dev))
    ct = OracleCostTracer(grids, A, horizon)
    ct.sim.load_state(pos, goal)
    stream = torch.from_numpy(targets).to(dev)
    cursor = torch.zeros((E, A), dtype=torch.int32, device=dev)
    best = torch.full_like(cursor, -1)
    reward, reached = torch.empty((E, A), device=dev), torch.empty((E, A), device=dev)
    obs = torch.empty((E, A, 2, 11, 11), device=dev)
    desc = type(builder._desc).from_buffer_copy(builder._desc)
    if not with_info:
        desc.agent_info = None
    lib, ref = builder._lib, ctypes.byref(desc)
    plain = set()
    rng = np.random.default_rng(5)
    for t in range(steps):
        builder.refresh_distances(sim.cur_x, sim.cur_y, sim.goal_x, sim.goal_y)
        assert lib.jl_costtracer_observe(sim._sim_ref, ref, best.data_ptr(), obs.data_ptr(), _stream(obs.device)) == 0
        ct.refresh_distances()
        want = ct.observe()
        got = obs.cpu().numpy()
        assert np.array_equal(got, want), f"t={t}: {np.argwhere(got != want)[:4].tolist()}"
        assert np.array_equal(best.cpu().numpy(), ct.best), t
        far = builder.cost_to_go.cpu().numpy().view(np.uint16).reshape(E, A, -1).astype(np.int32)
        plain.add(tuple(((far < 0xFFFF) & (far > 4080)).any(-1)[2].tolist()))
        sim.update_actions(torch.from_numpy(acts).to(dev))
        sim.step_sim_only()
        assert lib.jl_costtracer_reward_goals(sim._sim_ref, ref, best.data_ptr(), stream.data_ptr(), horizon + 1,
                                              cursor.data_ptr(), reward.data_ptr(), reached.data_ptr(),
                                              _stream(obs.device)) == 0
        ct.step(acts, targets)
        assert np.array_equal(reward.cpu().numpy(), ct.rewards), t
        assert np.array_equal(reached.cpu().numpy(), ct.reached), t
        assert np.array_equal(cursor.cpu().numpy(), ct.cursor), t
        if t == 0:
            assert ct.reached.all()
        acts = rng.integers(0, 5, size=(E, A)).astype(np.uint8)
    # the third map's fields were of both kinds at once, and changed kind
    assert len(plain) > 1 and all(any(p) and not all(p) for p in plain)
