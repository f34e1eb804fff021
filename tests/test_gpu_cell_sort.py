"""GPU parity of the small-flock sort (workgroups that each own a range of
cells): sorted pairs, cell ranges, sorted state and lists of one step are the
oracle's bits at the sizes where it changes method: lists ranked by counting
(512), the bitonic network's powers of two, more agents than a workgroup holds
(4,096) spread over cells or in one cell, the largest flock and grid it takes
and the next ones up (the radix sort's)."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.engine import Batch, Flock
from behavert_amd.types import GridParams, ProxParams

from ._parity import dev, empty_u32, first_mismatch, oracle_grid_outputs, u32

pytestmark = pytest.mark.gpu


def flock_state(seed, xyz):
    rng = np.random.default_rng(seed)
    return W.make_state(np.asarray(xyz, np.float32), *W.directions_and_speeds(rng, len(xyz)))


def check(ctx, orc, grid, st, K=4):
    prox = ProxParams.make(K, 4.0)
    fl = Flock(ctx, grid, prox, W.plain_steer(), st)
    fl.step(0.05, 0)
    got, want = fl.grid_outputs(), oracle_grid_outputs(orc, grid, prox, st)
    for k in ("hash", "cell_start", "cell_end", "sorted_pos", "sorted_forward", "sorted_smooth_accel", "lists"):
        assert first_mismatch(got[k].view(np.uint32), want[k].view(np.uint32)) is None, k
    alone = empty_u32(len(st["pos"]), 2)
    ctx.hash_sort(grid, dev(st["pos"]), alone)
    assert first_mismatch(u32(alone), want["hash"]) is None


@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 511, 512, 513, 1023, 1024])
def test_one_group_of_m_agents(ctx, orc, m):
    """Grid of one cell: every agent in one workgroup."""
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (1, 1, 1))
    check(ctx, orc, grid, flock_state(m, np.random.default_rng(m).uniform(0, 4, (m, 3))))


@pytest.mark.parametrize("m", [1025, 2047, 2048, 2049, 4095, 4096, 4097, 20000])
@pytest.mark.parametrize("cells", [1, 3, 40])
def test_crowded_cells_of_a_larger_grid(ctx, orc, m, cells):
    """m agents in the first cells of a 16 x 16 x 9 grid (nine per workgroup)
    and 3,000 anywhere, in shuffled ID order."""
    rng = np.random.default_rng(m + cells)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (16, 16, 9))
    at = np.c_[4.0 * (np.arange(m) % cells % 16), 4.0 * (np.arange(m) % cells // 16), np.zeros(m)]
    xyz = np.concatenate([at + rng.uniform(0, 3.9, (m, 3)), rng.uniform(0, 1, (3000, 3)) * (64.0, 64.0, 36.0)])
    check(ctx, orc, grid, flock_state(m, xyz[rng.permutation(len(xyz))]))


@pytest.mark.parametrize("n,size", [((1 << 17), (128, 64, 128)), ((1 << 17) + 1, (64, 64, 64)),
                                    (70001, (128, 64, 128)), (70001, (128, 64, 129)), (4097, (4, 1, 1))])
def test_limits(ctx, orc, n, size):
    rng = np.random.default_rng(n)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, size)
    check(ctx, orc, grid, flock_state(n, rng.uniform(-2.0, 2.0, (n, 3)) + rng.uniform(0, 1, (n, 3)) * 4.0 * np.array(size)))


def test_small_batch(ctx, orc):
    """A batch below the limit: each flock equals the oracle's own step."""
    grids = [W.cube_grid(20.0), W.cube_grid(36.0), W.cube_grid(8.0)]
    sizes, sides = [700, 1500, 65], [20.0, 36.0, 8.0]
    states = [W.uniform_flock(n, s, i) for i, (n, s) in enumerate(zip(sizes, sides))]
    weights = np.full((3, 3), 0.7, np.float32)
    state = {k: np.concatenate([s[k] for s in states]) for k in states[0]}
    prox, steer = ProxParams.make(16, 4.0), W.plain_steer((0.7, 0.7, 0.7))
    b = Batch(ctx, grids, sizes, weights, prox, steer, state)
    hosts = [orc.HostFlock(g, prox, s) for g, s in zip(grids, states)]
    for step in range(3):
        b.step(0.05, step)
        for h in hosts:
            h.step(steer, 0.05, step)
    got = b.state()
    for f, h in enumerate(hosts):
        for k in ("pos", "forward", "smooth_accel"):
            assert first_mismatch(got[k][b.flock_slice(f)].view(np.uint32), getattr(h, k).view(np.uint32)) is None
