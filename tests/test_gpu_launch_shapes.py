"""The rules that choose how a call's work is cut into workgroups keep to the
bounds that they are there for (read off the launches of a captured call)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

LDS = 160 * 1024


def cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def state_build(E, A, W, H):
    """A builder on open maps whose fields are there, its next build's launches."""
    from iclr_2027_jointoom_amd import profile
    from launches import launches

    rng = np.random.default_rng(E + A)
    b = profile(W, H).MapfGPTObservationBuilder(torch.zeros((E, W, H), dtype=torch.int32, device="cuda"), A)
    st = [torch.from_numpy(rng.integers(0, n, (E, A)).astype(np.int16)).cuda() for n in (W, H, W, H)]
    b.build_tokens_from_state(*st)
    torch.cuda.synchronize()
    return launches(lambda: b.build_tokens_from_state(*st))


@pytest.mark.parametrize("W,H", [(96, 96), (130, 192)])
@pytest.mark.parametrize("E,A", [(1, 1), (3, 600), (16, 512), (64, 128), (100, 100), (130, 128), (200, 64), (300, 100),
                                 (150, 200), (300, 33), (600, 40)])
def test_token_slices_run_at_once(E, A, W, H):
    """Slices of an env's egos are cut smaller only while all of them are
    resident at once: a second round costs what the smaller slices save."""
    got = [k for k in state_build(E, A, W, H) if "tokens_kernel" in k.name]
    assert len(got) == 1
    whole = E * -(-A // 512)  # no slice cut
    assert got[0].groups <= max(whole, cus() * min(2, LDS // got[0].lds)), got


@pytest.mark.parametrize("W,H", [(65, 160), (128, 192), (160, 224), (208, 224), (96, 256), (128, 256), (200, 256), (256, 256)])
def test_split_searches_run_at_once(W, H):
    """A map split over the wavefronts of a workgroup: the workgroups' LDS
    leaves room for as many per CU as the launch counts on."""
    E, A = 20, 256
    got = [k for k in state_build(E, A, W, H) if "unpack_fields_kernel" in k.name]
    assert len(got) == 1
    assert got[0].groups <= cus() * (LDS // got[0].lds), got
    # and for at least 12 of a CU's 16 wavefronts (five-wavefront groups: 15)
    assert (LDS // got[0].lds) * got[0].threads >= 12 * 64, got


# both sides of every line of the rule, and what small envs of a raw-row build take
@pytest.mark.parametrize("E,A,rows,threads", [(1, 16, 0, 512), (1, 17, 0, 1024), (256, 33, 0, 1024), (257, 64, 0, 512),
                                              (257, 65, 0, 1024), (257, 33, 1, 1024), (512, 65, 0, 1024),
                                              (513, 65, 0, 512), (513, 65, 1, 512), (700, 513, 0, 1024)])
def test_single_launch_workgroup_size(E, A, rows, threads):
    """1,024 threads where an env has a CU of its own; where two envs share
    one, only for envs large enough to gain from it, or raw rows."""
    from iclr_2027_jointoom_amd import profile
    from launches import launches

    if cus() != 256:
        pytest.skip("sizes of a card of 256 CUs")
    b = profile(32, 32).MapfGPTObservationBuilder(torch.zeros((E, 32, 32), dtype=torch.int32, device="cuda"), A)
    st = [torch.zeros((E, A), dtype=torch.int16, device="cuda")] * 4
    raw = torch.zeros((E * A, 13), dtype=torch.int16, device="cuda")
    call = (lambda: b.build_tokens(raw)) if rows else (lambda: b.build_tokens_from_state(*st))
    call()
    torch.cuda.synchronize()
    got = [k for k in launches(call) if "build_kernel" in k.name]
    assert len(got) == 1 and b.single_launch
    assert (got[0].groups, got[0].threads) == (E, threads), got


@pytest.mark.parametrize("E,A", [(1, 1), (148, 16), (200, 30), (239, 9), (4, 48), (250, 64), (300, 20)])
def test_node_workgroups_all_have_rows(E, A):
    """An env of at most 64 agents has no node workgroup without an agent
    (every second one idle would leave half of the XCDs idle)."""
    from iclr_2027_jointoom_amd import profile
    from launches import launches

    sim = profile(64, 64).GridWorldSimulator(torch.zeros((E, 64, 64), dtype=torch.int32, device="cuda"), A, 0,
                                             E * 4096, 1, "standard_mapf", 64)
    got = [k for k in launches(sim.build_magat_plus_nodes) if "nodes_kernel" in k.name]
    assert len(got) == 1
    # E workgroups of all A agents, or of a power of two of them, 4 to 32
    assert got[0].groups in [E * -(-A // n) for n in (64, 32, 16, 8, 4)], got
