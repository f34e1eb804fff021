"""GPU parity of the small-flock sort for flocks gathered in few cells, whose crowded
ranges are cut into chunks that several workgroups sort: sorted pairs, cell ranges,
sorted state and lists are the oracle's bits, at the sizes around which a range becomes
crowded (2,048), for one, several and all ranges crowded, for IDs in any order, in order
of place and in runs, with NaN positions among them, and for a batch."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.engine import Batch
from behavert_amd.types import GridParams, ProxParams

from ._parity import dev, empty_u32, first_mismatch, u32
from .test_gpu_cell_sort import check, flock_state

pytestmark = pytest.mark.gpu


def gathered(rng, n, side, at=80.0, cell=4.0):
    """n positions in side^3 cells of the given size from `at` on."""
    return at + rng.uniform(0.0, 0.9999 * cell * side, (n, 3))


def ordered(rng, xyz, order, cell=4.0):
    if order == "random":
        return xyz[rng.permutation(len(xyz))]
    key = np.floor(xyz / cell).astype(np.int64)
    xyz = xyz[np.lexsort((key[:, 0], key[:, 1], key[:, 2]))]
    if order == "place":
        return xyz
    runs = np.array_split(np.arange(len(xyz)), 31)  # of neighbouring cells, in turn
    return xyz[np.concatenate([r[rng.permutation(len(r))] for r in (runs[k] for k in rng.permutation(31))])]


def check_sort(ctx, orc, grid, st):
    want = orc.sort_radix(orc.calc_hash(grid, st["pos"]), grid.num_cells)
    got = empty_u32(len(st["pos"]), 2)
    ctx.hash_sort(grid, dev(st["pos"]), got)
    assert first_mismatch(u32(got), want) is None


@pytest.mark.parametrize("n", [2047, 2049, 3071, 4097, 8191, 20000])
@pytest.mark.parametrize("side", [1, 2, 5])
def test_gathered_flocks(ctx, orc, n, side):
    rng = np.random.default_rng(n + side)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (64,) * 3)
    # no more per cell than the oracle's scan of all pairs does in a second
    if n // side**3 <= 4097:
        check(ctx, orc, grid, flock_state(n, gathered(rng, n, side)))
    else:
        check_sort(ctx, orc, grid, flock_state(n, gathered(rng, n, side)))


@pytest.mark.parametrize("order", ["random", "place", "runs"])
@pytest.mark.parametrize("n,side", [(50000, 1), (50000, 3), (1 << 17, 1), (1 << 17, 2), ((1 << 17) - 3, 6), (1 << 17, 13)])
def test_order_of_ids(ctx, orc, n, side, order):
    rng = np.random.default_rng(n + side)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (64,) * 3)
    check_sort(ctx, orc, grid, flock_state(n, ordered(rng, gathered(rng, n, side), order)))


@pytest.mark.parametrize("size", [(100, 100, 100), (64, 64, 256), (33, 7, 1), (300, 1, 1)])
@pytest.mark.parametrize("sigma", [1.0, 6.0])
def test_blobs_beside_even_agents(ctx, orc, size, sigma):
    """Three blobs of unlike sizes, the rest anywhere, a few with NaN positions."""
    rng = np.random.default_rng(size[0])
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, size)
    far = 4.0 * np.array(size)
    xyz = np.concatenate([c * far + sigma * rng.standard_normal((m, 3))
                          for c, m in ((0.2, 20000), (0.5, 5000), (0.9, 2500))] + [rng.uniform(0, 1, (9001, 3)) * far])
    st = flock_state(len(xyz), xyz[rng.permutation(len(xyz))])
    st["pos"][::4001, :3] = np.nan
    check_sort(ctx, orc, grid, st)


@pytest.mark.parametrize("n,side,blobs", [(47839, 140.0, 2), (100517, 184.0, 6)])
@pytest.mark.parametrize("seed", [16, 21, 22, 23])
def test_ranges_on_either_side_of_the_sample(ctx, orc, n, side, blobs, seed):
    """Ranges of about 2,048 agents, which the sampled keys show crowded or light by
    chance: the workgroup of one that they show light is counted on as a helper."""
    rng = np.random.default_rng(seed)
    centres = rng.random((blobs, 3)) * side
    of = rng.permutation(n) % blobs
    xyz = side - np.abs(side - np.abs(centres[of] + 10.0 * rng.standard_normal((n, 3))))
    check_sort(ctx, orc, W.cube_grid(side), flock_state(n, np.clip(xyz, 0.0, np.nextafter(np.float32(side), 0))))


@pytest.mark.parametrize("n,m", [(16384, 2048), (16384, 2049), (16385, 2049), (16385, 4096), (16385, 4097), (60000, 4097),
                                 (60000, 3100)])
def test_one_range_around_the_limits(ctx, orc, n, m):
    """A range of m agents in three cells, the others anywhere: whether it is crowded
    depends on m and on the flock's size."""
    rng = np.random.default_rng(n + m)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (64, 64, 16))  # 256 cells, four rows, per workgroup
    xyz = rng.uniform(0, 1, (n - m, 3)) * (256.0, 256.0, 64.0)
    inside = (xyz[:, 1] // 16 == 6) & (xyz[:, 2] // 4 == 5)
    xyz[inside, 2] += 4.0
    own = np.c_[rng.integers(9, 12, m) * 4.0, np.full(m, 100.0), np.full(m, 20.0)] + rng.uniform(0, 3.9, (m, 3))
    xyz = np.concatenate([own, xyz])
    check_sort(ctx, orc, grid, flock_state(n, xyz[rng.permutation(n)]))


def test_two_crowded_cells_and_their_neighbours(ctx, orc):
    """Whole steps, with the gathers of the sorted state and the lists."""
    rng = np.random.default_rng(5)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (64,) * 3)
    xyz = np.concatenate([gathered(rng, 3000, 1, 16.0), gathered(rng, 4500, 1, 200.0), rng.uniform(0, 256, (60000, 3))])
    check(ctx, orc, grid, flock_state(len(xyz), xyz[rng.permutation(len(xyz))]), K=16)


def test_crowded_flock_of_a_batch(ctx, orc):
    grids = [W.cube_grid(40.0), W.cube_grid(20.0), W.cube_grid(60.0)]
    sizes = [3000, 700, 5000]
    rng = np.random.default_rng(6)
    states = [W.uniform_flock(n, s, i) for i, (n, s) in enumerate(zip(sizes, (40.0, 20.0, 60.0)))]
    states[2]["pos"][:, :3] = rng.uniform(0.0, 8.0, (5000, 3))
    weights = np.full((3, 3), 0.7, np.float32)
    state = {k: np.concatenate([s[k] for s in states]) for k in states[0]}
    prox, steer = ProxParams.make(16, 4.0), W.plain_steer((0.7, 0.7, 0.7))
    b = Batch(ctx, grids, sizes, weights, prox, steer, state)
    hosts = [orc.HostFlock(g, prox, s) for g, s in zip(grids, states)]
    for step in range(2):
        b.step(0.05, step)
        for h in hosts:
            h.step(steer, 0.05, step)
    got = b.state()
    for f, h in enumerate(hosts):
        for k in ("pos", "forward", "smooth_accel"):
            assert first_mismatch(got[k][b.flock_slice(f)].view(np.uint32), getattr(h, k).view(np.uint32)) is None
