"""The automatic launch shapes beyond K = 32 on both sides of their rules (K 80
and 81, crowded grids and sparse ones, with and without the feature update, the
list call alone): bit-exact against the CPU oracle."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.engine import Flock
from behavert_amd.types import ProxParams

from ._parity import dev, empty_u32, first_mismatch, oracle_grid_outputs, u32

pytestmark = pytest.mark.gpu

N = (1 << 17) + 77  # above the four-lane kernels


@pytest.mark.parametrize("K", [33, 48, 64, 80, 81])
@pytest.mark.parametrize("side,crowded", [(200.0, False), (96.0, True)])
@pytest.mark.parametrize("features", [False, True])
def test_shapes(ctx, orc, K, side, crowded, features):
    grid, prox = W.cube_grid(side), ProxParams.make(K, 4.0)
    assert (N // 8 >= grid.num_cells) == crowded
    st = W.uniform_flock(N, side, K)
    f = np.random.default_rng(K).uniform(0, 1, (N, 4)).astype(np.float32) if features else None
    rate = 0.1 if features else 0.0
    fl = Flock(ctx, grid, prox, W.plain_steer(), st, features=f, sorted_smooth_accel=False)
    hf = orc.HostFlock(grid, prox, st, features=f)
    fl.step(0.05, 0, rate)
    hf.step(W.plain_steer(), 0.05, 0, rate)
    assert first_mismatch(u32(fl.lists), hf.lists) is None
    got = fl.state()
    for k in ("pos", "forward", "smooth_accel"):
        assert first_mismatch(got[k].view(np.uint32), getattr(hf, k).view(np.uint32)) is None, k
    if features:
        assert first_mismatch(u32(fl.features), hf.features.view(np.uint32)) is None
    else:
        o = oracle_grid_outputs(orc, grid, prox, st)
        lists = empty_u32(N, 4 * (K // 4 + 1)).fill_(0x5A5A5A5A)
        ctx.neighbors(grid, prox, dev(o["sorted_pos"]), *[dev(o[k].view(np.int32)) for k in
                                                          ("hash", "cell_start", "cell_end")], lists)
        assert first_mismatch(u32(lists), o["lists"]) is None
