"""GPU parity of KNN lists (useKnn), whose entries depend on every accepted
candidate in order: bit-exact against the CPU oracle over caps (one lane per
agent up to the widest lists, which share a wave between fewer lanes), sparse
and crowded cells (rounds of 4 and 8, the log worked off many times), ties,
agents outside the grid and per-cell limits; and at 2^24 agents, where the log
holds whole indices."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.engine import Flock
from behavert_amd.types import GridParams, ProxParams

from ._parity import dev, empty_u32, first_mismatch, oracle_grid_outputs, u32

pytestmark = pytest.mark.gpu


def check(ctx, orc, grid, K, xyz, seed):
    rng = np.random.default_rng(seed)
    st = W.make_state(np.asarray(xyz, np.float32), *W.directions_and_speeds(rng, len(xyz)))
    prox = ProxParams.make(K, 4.0, use_knn=True)
    o = oracle_grid_outputs(orc, grid, prox, st)
    lists = empty_u32(len(xyz), 4 * (K // 4 + 1)).fill_(0x5A5A5A5A)
    ctx.neighbors(grid, prox, dev(o["sorted_pos"]), *[dev(o[k].view(np.int32)) for k in
                                                      ("hash", "cell_start", "cell_end")], lists)
    assert first_mismatch(u32(lists), o["lists"]) is None
    return o["lists"]


@pytest.mark.parametrize("K", [1, 2, 7, 16, 32, 33, 64, 129, 252])
@pytest.mark.parametrize("per_cell", [1, 4, 40])
def test_caps_and_densities(ctx, orc, K, per_cell):
    rng = np.random.default_rng(K)
    n = 64 * per_cell * 4 + 37
    side = 4.0 * round((n / per_cell) ** (1.0 / 3.0))
    lists = check(ctx, orc, W.cube_grid(side), K, rng.uniform(0, side, (n, 3)), K)
    if per_cell == 40 and K <= 33:
        assert (lists[:, 0] == K).mean() > 0.5  # entries are replaced


@pytest.mark.parametrize("max_bodies", [0xFFFFFFFF, 3])
def test_ties_outside_and_limits(ctx, orc, max_bodies):
    """Positions on a half-unit lattice (equal distances), some outside the grid."""
    rng = np.random.default_rng(3)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (6, 2, 5), max_bodies=max_bodies)
    xyz = 0.5 * rng.integers(-8, 48, (4000, 3)) * np.array([1.0, 0.4, 0.9])
    xyz[::50, 0] = np.nan
    check(ctx, orc, grid, 12, xyz, 3)


def test_indices_beyond_24_bits(ctx):
    """2^24 + 37 agents, lists never full: equal to the plain lists."""
    n = (1 << 24) + 37
    side = 4.0 * 330
    g = torch.Generator(device="cuda").manual_seed(1)
    pos = torch.rand(n, 4, generator=g, device="cuda") * side
    zero = np.zeros((n, 4), np.float32)
    prox = ProxParams.make(31, 4.0)
    fl = Flock(ctx, W.cube_grid(side), prox, W.plain_steer(), {"pos": zero, "forward": zero, "smooth_accel": zero})
    fl.pos.copy_(pos)
    fl.reorder_sim_data()
    fl.compute_neighborhoods()
    plain = fl.lists.clone()
    assert int(plain[:, 0].max()) < 31
    fl.prox = ProxParams.make(31, 4.0, use_knn=True)
    fl.compute_neighborhoods()
    assert torch.equal(plain, fl.lists)
