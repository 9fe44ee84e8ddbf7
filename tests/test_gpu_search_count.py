"""The row search's count of levels of more than a limit of cells (the
builder's diagnostics[0] with its limit of 4,096), on every layout, unsplit
ones too, with a limit of 40 cells (jl_search_count in libjl_bench.so)."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

LIMIT = 40


@pytest.mark.parametrize("W,H", [(64, 64), (65, 64), (129, 64), (256, 64), (64, 96), (127, 96), (200, 96), (33, 128),
                                 (128, 128), (129, 128), (64, 256), (65, 256), (256, 256)])
def test_cells_past_the_limit(oracle, W, H):
    from bench import load_probe
    from iclr_2027_jointoom_amd._abi import check

    count = load_probe().jl_search_count
    count.argtypes = [ctypes.c_void_p] + [ctypes.c_int32] * 4 + [ctypes.c_void_p] * 2
    rng = np.random.default_rng(W * 5 + H)
    out = torch.zeros(1, dtype=torch.int32, device="cuda")
    some = 0
    for density in (0.0, 0.1, 0.3, 0.45):
        grid = (rng.random((W, H)) < density).astype(np.uint8)
        free = np.argwhere(grid == 0)
        bits = torch.from_numpy(oracle.encode(grid[None])[0].view(np.int32).copy()).cuda()
        for goal in (free[0], free[-1], free[len(free) // 2], free[rng.integers(len(free))]):
            field = oracle.bfs_u16(grid, goal)[0].astype(np.int64)
            cells = np.bincount(field[field < 0xFFFF])
            check(count(bits.data_ptr(), W, H, int(goal[0]), int(goal[1]), out.data_ptr(),
                        torch.cuda.current_stream().cuda_stream), "search count")
            want = int(np.maximum(0, cells - LIMIT).sum())
            assert int(out.item()) == want, (density, goal.tolist())
            some += want > 0
    assert some >= 4
