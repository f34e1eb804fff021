"""GPU parity of the list call where the first wave of a workgroup scans sparse rows
for all its agents and four lanes each take the rest: launch sizes on both sides
of each rule, tails of a workgroup of every kind, flocks whose density rises from
one to sixty per cell along x, agents outside the grid, caps that fill in the
first cells and ones that never fill.  Lists are whole numbers: bit-exact against
the CPU oracle."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.types import GridParams, ProxParams

from ._parity import dev, empty_u32, first_mismatch, oracle_grid_outputs, u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 8, 16, 32, 64, 252])
@pytest.mark.parametrize("n,max_bodies", [(49152, 0xFFFFFFFF), (49153, 0xFFFFFFFF), (60000 - 17, 0xFFFFFFFF),
                                          (32768, 0xFFFFFFFF), (32769, 0xFFFFFFFF), (90112, 0xFFFFFFFF),
                                          (90113, 0xFFFFFFFF), (60000, 9)])
@pytest.mark.parametrize("sparse", [False, True])
def test_lists(ctx, orc, K, n, max_bodies, sparse):
    rng = np.random.default_rng(K + n)
    size = np.array((44, 40, 37) if sparse else (30, 24, 12))
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, size, max_bodies=max_bodies)
    xyz = rng.uniform(0, 1, (n, 3)) ** (1.0 if sparse else (0.35, 1.0, 1.0)) * (4.0 * size)
    xyz[::1009] = rng.uniform(-9.0, 4.0 * size + 9.0, xyz[::1009].shape)
    st = W.make_state(xyz.astype(np.float32), *W.directions_and_speeds(rng, n))
    prox = ProxParams.make(K, 4.0)
    o = oracle_grid_outputs(orc, grid, prox, st)
    lists = empty_u32(n, 4 * (K // 4 + 1)).fill_(0x5A5A5A5A)
    ctx.neighbors(grid, prox, dev(o["sorted_pos"]), *[dev(o[k].view(np.int32)) for k in
                                                      ("hash", "cell_start", "cell_end")], lists)
    assert first_mismatch(u32(lists), o["lists"]) is None


@pytest.mark.parametrize("n,K", [(106496, 16), (106497, 16), (106496, 32), (49152, 15), (49153, 15), (16384, 8),
                                 (16385, 8), (16385, 4)])
def test_lists_at_the_lines_by_size(ctx, orc, n, K):
    """Crowded and sparse flocks at the sizes where the quads, or their limit of the
    row scan (more than four per cell on average), begin or end."""
    test_lists(ctx, orc, K, n, 0xFFFFFFFF, True)
    test_lists(ctx, orc, K, n, 0xFFFFFFFF, False)
    test_lists(ctx, orc, K, n - n % 64 + 1, 0xFFFFFFFF, False)
