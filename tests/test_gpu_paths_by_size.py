"""Paths that a call reaches by its size, where the small flocks of other tests take
another one: two radix-sorted steps of different sizes on one context, the batch's
radix sort with features and wander, and four lanes per agent with NaN, coincident and
out-of-grid agents."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.engine import Context, Flock
from behavert_amd.types import GridParams, ProxParams

from ._parity import first_mismatch, oracle_grid_outputs
from .test_gpu_batch import compare_flocks, run_pair, small_batch
from .test_gpu_proximity import gpu_lists

pytestmark = pytest.mark.gpu

RADIX = (1 << 17) + 1  # agents from which the radix sort runs


def test_radix_steps_of_two_sizes_on_one_context():
    flocks = []
    shared = Context(0)
    for n, side in ((3 * RADIX, 180.0), (RADIX, 120.0)):
        st, grid, prox = W.uniform_flock(n, side, n), W.cube_grid(side), ProxParams.make(8, 4.0)
        flocks.append((Flock(shared, grid, prox, W.plain_steer(), st),
                       Flock(Context(0), grid, prox, W.plain_steer(), st)))
    for step, k in enumerate((0, 1, 0, 1, 1, 0, 0)):
        for fl in flocks[k]:
            fl.step(0.05, step)
        a, b = flocks[k]
        for key, x in a.grid_outputs().items():
            assert first_mismatch(x.view(np.uint32), b.grid_outputs()[key].view(np.uint32)) is None, (step, key)
        for key, x in a.state().items():
            assert first_mismatch(x.view(np.uint32), b.state()[key].view(np.uint32)) is None, (step, key)


@pytest.mark.parametrize("K", [16, 40])
def test_radix_batch_with_wander_and_features(ctx, K):
    sizes, grids, weights, states, prox = small_batch(seed=3, sizes=(70000, 1, 0, 50001, 777, 20000), K=K)
    assert sum(int(n) for n in sizes) >= RADIX
    steer = W.plain_steer()
    steer.wander_weight = 0.3
    steer.wander_seed = 77
    g = np.random.default_rng(4)
    wander = [g.uniform(-1, 1, (int(n), 2)).astype(np.float32) for n in sizes]
    features = [g.random((int(n), 4), np.float32) for n in sizes]
    b, flocks = run_pair(ctx, sizes, grids, weights, states, prox, steps=3, base_steer=steer, wander=wander,
                         feature_rate=0.1, features=features)
    compare_flocks(b, flocks, grids)
    for f, fl in enumerate(flocks):
        if fl is None:
            continue
        for k in ("wander", "features"):
            got = getattr(b, k).cpu().numpy()[b.flock_slice(f)]
            assert first_mismatch(got.view(np.uint32), fl.state()[k].view(np.uint32)) is None, (f, k)
    b.close()


@pytest.mark.parametrize("maxb", [0xFFFFFFFF, 3])
@pytest.mark.parametrize("K", [4, 12, 32, 64])
def test_four_lanes_with_nan_and_coincident_agents(ctx, orc, K, maxb):
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (8,) * 3, max_bodies=maxb)
    prox = ProxParams.make(K, 4.0)
    rng = np.random.default_rng(K)
    xyz = rng.uniform(-6, 38, (6000, 3)).astype(np.float32)
    xyz[::500] = [np.nan, 2, 2]
    xyz[1::900] = [5.0, 5.0, 5.0]
    xyz[2] = [-1000.0, 9, 9]
    st = W.make_state(xyz, *W.directions_and_speeds(rng, len(xyz)))
    assert ctx.step_shape_for(prox, len(xyz), grid.num_cells)[2] == 4
    o = oracle_grid_outputs(orc, grid, prox, st)
    assert first_mismatch(gpu_lists(ctx, grid, prox, o), o["lists"]) is None
    fl, host = Flock(ctx, grid, prox, W.plain_steer(), st), orc.HostFlock(grid, prox, st)
    for step in range(2):
        fl.step(0.05, step)
        host.step(W.plain_steer(), 0.05, step)
        assert first_mismatch(fl.grid_outputs()["lists"].view(np.uint32), host.lists) is None, step
        got, want = fl.state(), host.state()
        for k in ("pos", "forward", "smooth_accel"):
            assert np.array_equal(got[k], want[k], equal_nan=True), (step, k)


@pytest.mark.parametrize("K", [27, 28, 56, 57, 80])
def test_crowded_fused_steps(ctx, orc, K):
    """About 20 agents per cell: quads of lanes visit their cells together or not, by K."""
    rng = np.random.default_rng(K)
    grid, prox = GridParams.direct((0.0,) * 3, (4.0,) * 3, (19,) * 3), ProxParams.make(K, 4.0)
    st = W.make_state(rng.uniform(0, 76, (RADIX, 3)).astype(np.float32), *W.directions_and_speeds(rng, RADIX))
    assert ctx.step_shape_for(prox, RADIX, grid.num_cells) == (True, True, 1)
    o = oracle_grid_outputs(orc, grid, prox, st)
    assert first_mismatch(gpu_lists(ctx, grid, prox, o), o["lists"]) is None
    fl, host = Flock(ctx, grid, prox, W.plain_steer(), st), orc.HostFlock(grid, prox, st)
    fl.step(0.05, 0)
    host.step(W.plain_steer(), 0.05, 0)
    assert first_mismatch(fl.grid_outputs()["lists"].view(np.uint32), host.lists) is None
    for k, x in fl.state().items():
        assert first_mismatch(x.view(np.uint32), host.state()[k].view(np.uint32)) is None, k
