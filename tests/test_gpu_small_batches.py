"""Batches of few envs, whose work is split further over the chip: the
single-launch build in 1,024-thread workgroups, the token pass in slices of
an env's egos, the node pass with a slice's rows shared out.  Sizes on both
sides of every split, against the C oracle (whole numbers and node features,
which are exact)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def world(E, W, H, A, seed):
    rng = np.random.default_rng(seed)
    grids = (rng.random((E, W, H)) < 0.1).astype(np.uint8)
    pos, goals = np.zeros((E, A, 2), np.int16), np.zeros((E, A, 2), np.int16)
    for e, g in enumerate(grids):
        free = np.argwhere(g == 0)
        pos[e] = free[rng.choice(len(free), A, replace=len(free) < A)]
        goals[e] = free[rng.choice(len(free), A)]
    return rng, grids, pos, goals


def builds_match(oracle, E, W, H, A, seed):
    """Every goal new, then a fifth of them, then none; tokens, state rows and diagnostics."""
    from iclr_2027_jointoom_amd import profile

    rng, grids, pos, goals = world(E, W, H, A, seed)
    builder = profile(W, H).MapfGPTObservationBuilder(torch.from_numpy(grids.astype(np.int32)).cuda(), A)
    ob = oracle.OracleMapfGPT(grids, A)
    for step in range(3):
        if step == 1:
            goals[rng.random((E, A)) < 0.2] = pos[0, 0]
        st = [np.ascontiguousarray(v) for v in (pos[..., 0], pos[..., 1], goals[..., 0], goals[..., 1])]
        builder.build_tokens_from_state(*(torch.from_numpy(v).cuda() for v in st))
        ob.build_state(*st)
        torch.cuda.synchronize()
        assert np.array_equal(builder.tokens.cpu().numpy(), ob.tokens), step
        assert np.array_equal(builder.state_packed.cpu().numpy().view(np.uint16), ob.state_packed), step
        assert builder.diagnostics.cpu().tolist() == ob.diagnostics.tolist(), step
    return builder


@pytest.mark.parametrize("E,A", [(1, 1), (1, 16), (1, 17), (2, 64), (1, 512), (3, 513), (512, 18), (513, 18)])
def test_single_launch_workgroups(oracle, E, A):
    assert builds_match(oracle, E, 32, 32, A, E + A).single_launch


@pytest.mark.parametrize("W,H,E,A", [(96, 96, 1, 1), (96, 96, 1, 32), (96, 96, 2, 33), (100, 64, 5, 65), (96, 96, 300, 33),
                                     (130, 192, 1, 513), (256, 256, 2, 127)])
def test_token_slices(oracle, W, H, E, A):
    assert not builds_match(oracle, E, W, H, A, W + A).single_launch


@pytest.mark.parametrize("E,A", [(1, 1), (1, 4), (3, 5), (1, 63), (2, 64), (2, 65), (5, 130), (1, 1025), (130, 70)])
def test_shared_node_slices(oracle, E, A):
    from iclr_2027_jointoom_amd import profile

    W, H = 64, 96
    _, grids, pos, goals = world(E, W, H, A, A * 3 + E)
    rows = np.zeros((E, A, 8), np.int16)
    rows[..., 0] = np.arange(E)[:, None]
    rows[..., 1] = np.arange(A)[None]
    rows[..., 2:4], rows[..., 4:6], rows[..., 7] = pos, goals, 1
    rows = rows.reshape(E * A, 8)
    sim = profile(W, H).StatelessGridWorldSimulator(torch.from_numpy(grids.astype(np.int32)).cuda(), A, 3)
    dev = torch.from_numpy(rows).cuda()
    sim.update_derived_state(dev, len(rows))
    sim.build_magat_plus_inputs(dev)
    m = oracle.OracleMagat(grids, A)
    m.update_energy(rows.view(np.uint16), len(rows))
    m.refresh(rows.view(np.uint16))
    m.nodes()
    m.edges()
    torch.cuda.synchronize()
    assert np.array_equal(sim.pyg_x.cpu().numpy(), m.pyg_x)
    ei, ea = m.valid_edges()
    assert int(sim.pyg_num_edges.item()) == ei.shape[1]
    assert np.array_equal(sim.pyg_edge_index.cpu().numpy(), ei)
    assert np.array_equal(sim.pyg_edge_attr.cpu().numpy(), ea)
