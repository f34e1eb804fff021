"""Lists of positions that have moved since the sort (the reorder gathers new
positions through the older permutation): an agent never enters its own list,
wherever its position lies, on both sides of 2^17 agents and with every way of
building the lists; KNN lists are the oracle's bits."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.types import OPT_LDS_LISTS, ProxParams

from ._parity import dev, empty_u32, first_mismatch, u32

pytestmark = pytest.mark.gpu


def moved(orc, n, per_cell, far, seed):
    """Grid, the sort of n agents, and their positions moved by up to a cell, one in 50 (far) anywhere."""
    rng = np.random.default_rng(seed)
    side = 4.0 * round((n / per_cell) ** (1.0 / 3.0))
    grid = W.cube_grid(side)
    old = W.uniform_flock(n, side, seed)["pos"]
    h = orc.sort_radix(orc.calc_hash(grid, old), grid.num_cells)
    new = old.copy()
    new[:, :3] += rng.uniform(-4.0, 4.0, (n, 3)).astype(np.float32)
    if far:
        new[::50, :3] = rng.uniform(-6.0, side + 6.0, new[::50, :3].shape)
    return grid, h, *orc.cell_ranges(h, grid.num_cells), orc.reorder(h, new)


def device_lists(ctx, grid, prox, h, s, e, spos):
    lists = empty_u32(len(spos), 4 * (prox.max_neighbors // 4 + 1)).fill_(0x5A5A5A5A)
    ctx.neighbors(grid, prox, dev(spos), dev(h.view(np.int32)), dev(s.view(np.int32)), dev(e.view(np.int32)), lists)
    return u32(lists)


@pytest.mark.parametrize("n,lds,knn", [(5003, -1, False), (5003, 1, False), (5003, 0, False),
                                       ((1 << 17) + 77, -1, False), (5003, -1, True)])
@pytest.mark.parametrize("per_cell", [1, 12])
@pytest.mark.parametrize("far", [False, True])
def test_no_agent_in_its_own_list(ctx, orc, n, lds, knn, per_cell, far):
    grid, h, s, e, spos = moved(orc, n, per_cell, far, n + per_cell)
    prox = ProxParams.make(16, 4.0, use_knn=knn)
    ctx.set_option(OPT_LDS_LISTS, lds)
    try:
        lists = device_lists(ctx, grid, prox, h, s, e, spos)
    finally:
        ctx.set_option(OPT_LDS_LISTS, -1)
    held = np.arange(16)[None, :] < lists[:, :1]
    assert held.any()
    assert not (held & (lists[:, 1:17] == np.arange(n, dtype=np.uint32)[:, None])).any()


@pytest.mark.parametrize("per_cell", [1, 5, 30])
@pytest.mark.parametrize("K", [4, 16])
@pytest.mark.parametrize("far", [False, True])
def test_knn_lists(ctx, orc, per_cell, K, far):
    grid, h, s, e, spos = moved(orc, 4099, per_cell, far, K + per_cell)
    prox = ProxParams.make(K, 4.0, use_knn=True)
    lists = device_lists(ctx, grid, prox, h, s, e, spos)
    assert first_mismatch(lists, orc.neighbors(grid, prox, spos, h, s, e)) is None
