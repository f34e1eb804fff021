"""GPU parity of the neighbour lists of sparse flocks, whose waves scan the
cells of a row as one run: grids of few cells along x, agents outside the grid,
runs around the longest that the scan takes, caps around the list head that it
stages, and launch sizes on both sides of the wide kernel's limit.  Lists are
whole numbers: bit-exact against the CPU oracle."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.engine import Flock
from behavert_amd.types import OPT_LDS_LISTS, GridParams, ProxParams

from ._parity import dev, empty_u32, first_mismatch, oracle_grid_outputs, u32

pytestmark = pytest.mark.gpu


def state(rng, xyz):
    return W.make_state(np.asarray(xyz, np.float32), *W.directions_and_speeds(rng, len(xyz)))


def check(ctx, orc, grid, K, st):
    prox = ProxParams.make(K, 4.0)
    o = oracle_grid_outputs(orc, grid, prox, st)
    args = [dev(o[k].view(np.int32)) for k in ("hash", "cell_start", "cell_end")]
    for mode in (1, 0):
        ctx.set_option(OPT_LDS_LISTS, mode)
        lists = empty_u32(len(st["pos"]), 4 * (K // 4 + 1)).fill_(0x5A5A5A5A)
        try:
            ctx.neighbors(grid, prox, dev(o["sorted_pos"]), *args, lists)
        finally:
            ctx.set_option(OPT_LDS_LISTS, -1)
        assert first_mismatch(u32(lists), o["lists"]) is None, f"lds_lists={mode}"
    return o


@pytest.mark.parametrize("size", [(2, 6, 6), (3, 3, 3), (4, 1, 9), (7, 5, 1), (40, 3, 11)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 700])
def test_small_grids_and_agents_outside(ctx, orc, size, n):
    rng = np.random.default_rng(n)
    grid = GridParams.direct((-3.0, 1.0, 2.0), (4.0,) * 3, size)
    lo = np.array([-3.0, 1.0, 2.0])
    xyz = rng.uniform(lo - 5.0, lo + 4.0 * np.array(size) + 5.0, (n, 3))
    xyz[:: 17] += 400.0  # far outside
    check(ctx, orc, grid, 16, state(rng, xyz))


@pytest.mark.parametrize("run", [4, 5, 30, 31, 32])
@pytest.mark.parametrize("K", [1, 18, 19, 20, 21, 64])
def test_run_lengths_and_list_heads(ctx, orc, run, K):
    """Runs of `run` agents in cells that are empty but for every third row, all
    within the radius of each other: lists of run - 1 entries, cut at K."""
    rng = np.random.default_rng(run)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (9, 9, 9))
    xyz = []
    for y in range(1, 9, 3):
        for z in range(1, 9, 3):
            # a third of the run in each of the cells x = 3, 4, 5
            x = 14.1 + np.linspace(0.0, 3.8, run)
            xyz.append(np.c_[x, np.full(run, 4.0 * y + 2.0), np.full(run, 4.0 * z + 2.0)])
    xyz = np.concatenate(xyz)
    o = check(ctx, orc, grid, K, state(rng, xyz[rng.permutation(len(xyz))]))
    assert o["lists"][:, 0].max() == min(K, run - 1)


@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17, (1 << 17) + 65])
def test_step_on_both_sides_of_the_wide_launch(ctx, orc, n):
    """One fused step of a flock of one agent per cell."""
    st = W.uniform_flock(n, 204.0, n)
    grid, prox = W.cube_grid(204.0), ProxParams.make(32, 4.0)
    fl = Flock(ctx, grid, prox, W.plain_steer(), st, sorted_smooth_accel=False)
    fl.step(0.05, 0)
    hf = orc.HostFlock(grid, prox, st)
    hf.step(W.plain_steer(), 0.05, 0)
    assert first_mismatch(u32(fl.lists), hf.lists) is None
    got = fl.state()
    for k in ("pos", "forward", "smooth_accel"):
        assert first_mismatch(got[k].view(np.uint32), getattr(hf, k).view(np.uint32)) is None, k
