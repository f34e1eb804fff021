"""GPU parity of the neighbour search with four lanes per agent (small
launches): lists and steps bit-exact against the CPU oracle for sparse waves
(row scan), crowded cells (rounds of 16 candidates that end in any lane's
part), runs around the longest that the row scan takes, caps that cut a round,
per-cell limits, grids of few cells along x, agents outside the grid, tails of
a wave and of a workgroup, and launch sizes on both sides of the limit."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.engine import Flock
from behavert_amd.types import OPT_LDS_LISTS, GridParams, ProxParams, SteerParams

from ._parity import dev, empty_u32, first_mismatch, oracle_grid_outputs, u32

pytestmark = pytest.mark.gpu


def state(rng, xyz):
    return W.make_state(np.asarray(xyz, np.float32), *W.directions_and_speeds(rng, len(xyz)))


def check(ctx, orc, grid, K, st, steer=None):
    """The list call, and a step (its lists and new state)."""
    prox = ProxParams.make(K, 4.0)
    o = oracle_grid_outputs(orc, grid, prox, st)
    args = [dev(o[k].view(np.int32)) for k in ("hash", "cell_start", "cell_end")]
    lists = empty_u32(len(st["pos"]), 4 * (K // 4 + 1)).fill_(0x5A5A5A5A)
    ctx.neighbors(grid, prox, dev(o["sorted_pos"]), *args, lists)
    assert first_mismatch(u32(lists), o["lists"]) is None
    steer = steer or W.plain_steer()
    wander = np.zeros((len(st["pos"]), 2), np.float32) if steer.wander_weight else None
    for sorted_sa in (False, True):
        fl = Flock(ctx, grid, prox, steer, st, wander=wander, sorted_smooth_accel=sorted_sa)
        hf = orc.HostFlock(grid, prox, st, wander=wander)
        fl.step(0.05, 0)
        hf.step(steer, 0.05, 0)
        assert first_mismatch(u32(fl.lists), hf.lists) is None
        got = fl.state()
        for k in ("pos", "forward", "smooth_accel"):
            assert first_mismatch(got[k].view(np.uint32), getattr(hf, k).view(np.uint32)) is None, k
    return o


@pytest.mark.parametrize("size", [(2, 6, 6), (3, 3, 3), (4, 1, 9), (7, 5, 1), (40, 3, 11)])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 700])
def test_small_grids_and_agents_outside(ctx, orc, size, n):
    rng = np.random.default_rng(n)
    lo = np.array([-3.0, 1.0, 2.0])
    grid = GridParams.direct(lo, (4.0,) * 3, size)
    xyz = rng.uniform(lo - 5.0, lo + 4.0 * np.array(size) + 5.0, (n, 3))
    xyz[:: 17] += 400.0  # far outside
    check(ctx, orc, grid, 16, state(rng, xyz))


@pytest.mark.parametrize("K", [1, 3, 16, 17, 32, 33, 64, 252])
@pytest.mark.parametrize("per_cell,max_bodies", [(1, 0xFFFFFFFF), (9, 0xFFFFFFFF), (17, 0xFFFFFFFF), (60, 0xFFFFFFFF),
                                                 (17, 5)])
def test_caps_densities_and_limits(ctx, orc, K, per_cell, max_bodies):
    rng = np.random.default_rng(K)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (5, 4, 6), max_bodies=max_bodies)
    n = 120 * per_cell + 3
    check(ctx, orc, grid, K, state(rng, rng.uniform(0.0, [20.0, 16.0, 24.0], (n, 3))))


@pytest.mark.parametrize("run", [4, 5, 30, 31, 32, 33])
@pytest.mark.parametrize("K", [18, 64])
def test_run_lengths(ctx, orc, run, K):
    """Runs of `run` agents within the radius of each other over the cells
    x = 3, 4, 5 of every third row: lists of run - 1 entries, cut at K."""
    rng = np.random.default_rng(run)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (9, 9, 9))
    x = 14.1 + np.linspace(0.0, 3.8, run)
    xyz = np.concatenate([np.c_[x, np.full(run, 4.0 * y + 2.0), np.full(run, 4.0 * z + 2.0)]
                          for y in range(1, 9, 3) for z in range(1, 9, 3)])
    o = check(ctx, orc, grid, K, state(rng, xyz[rng.permutation(len(xyz))]))
    assert o["lists"][:, 0].max() == min(K, run - 1)


def test_step_options(ctx, orc):
    """Targets, wander and unequal sensing per behaviour."""
    rng = np.random.default_rng(5)
    steer = SteerParams.make(weights=(1.0, 0.8, 0.6), targets=W.moving_targets(0.3, 12.0), target_weight=0.4)
    steer.wander_weight = 0.3
    steer.alignment[1] = 3.0
    steer.cohesion[2] = 0.2
    check(ctx, orc, W.cube_grid(40.0), 32, state(rng, rng.uniform(0.0, 40.0, (3001, 3))), steer)


@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17, (1 << 17) + 1])
@pytest.mark.parametrize("side", [204.0, 96.0])
def test_both_sides_of_the_limit(ctx, orc, n, side):
    grid, prox = W.cube_grid(side), ProxParams.make(20, 4.0)
    st = W.uniform_flock(n, side, n)
    fl = Flock(ctx, grid, prox, W.plain_steer(), st, sorted_smooth_accel=False)
    fl.step(0.05, 0)
    hf = orc.HostFlock(grid, prox, st)
    hf.step(W.plain_steer(), 0.05, 0)
    assert first_mismatch(u32(fl.lists), hf.lists) is None
    got = fl.state()
    for k in ("pos", "forward", "smooth_accel"):
        assert first_mismatch(got[k].view(np.uint32), getattr(hf, k).view(np.uint32)) is None, k


@pytest.mark.parametrize("K", [27, 28, 32])
@pytest.mark.parametrize("per_cell,max_bodies", [(9, 0xFFFFFFFF), (30, 0xFFFFFFFF), (30, 7)])
def test_one_lane_scans_in_step(ctx, orc, K, per_cell, max_bodies):
    """The one-lane kernel's crowded waves, whose quads walk the same cells from
    K 28 on where they share one: quads that span cells, a tail of three lanes,
    agents outside the grid among them."""
    rng = np.random.default_rng(K + per_cell)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (5, 4, 6), max_bodies=max_bodies)
    xyz = rng.uniform(-1.0, [21.0, 17.0, 25.0], (120 * per_cell // 64 * 64 + 3, 3))
    ctx.set_option(OPT_LDS_LISTS, 1)
    try:
        check(ctx, orc, grid, K, state(rng, xyz))
    finally:
        ctx.set_option(OPT_LDS_LISTS, -1)
