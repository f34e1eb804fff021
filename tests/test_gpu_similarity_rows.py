"""Where the similarity passes store their rows: 16 bytes per lane where the array
allows it, whole rows and partial ones, nothing outside them; alone and with the
cluster steering, bit-exact against the CPU oracle."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.types import BcParams, GridParams, ProxParams, SteerParams

from ._parity import dev, empty_f32, f32, first_mismatch, oracle_grid_outputs

pytestmark = pytest.mark.gpu


def crowded(orc, n, K, seed):
    """A third of the agents in one corner: short lists and full ones."""
    rng = np.random.default_rng(seed)
    xyz = rng.uniform(0, 24, (n, 3))
    xyz[::3] *= 0.25
    st = W.make_state(xyz.astype(np.float32), *W.directions_and_speeds(rng, n))
    prox = ProxParams.make(K, 4.0)
    return rng, prox, oracle_grid_outputs(orc, GridParams.direct((0.0,) * 3, (4.0,) * 3, (6,) * 3), prox, st)


def same(a, b):
    return first_mismatch(f32(a).view(np.uint32), np.ascontiguousarray(b, np.float32).view(np.uint32)) is None


@pytest.mark.parametrize("K", [1, 3, 4, 31, 32, 35, 36, 100])
@pytest.mark.parametrize("n", [1, 64, 131, 1001])
@pytest.mark.parametrize("shift", [0, 1])
def test_rows(ctx, orc, K, n, shift):
    rng, prox, o = crowded(orc, n, K, 7 * K + n)
    feats = rng.standard_normal((n, 6)).astype(np.float32)
    stats = np.sort(rng.uniform(0, 1, (n, 4)), axis=1).astype(np.float32)
    f0 = rng.standard_normal((n, 4)).astype(np.float32)
    bc, sp = BcParams.make(6), SteerParams.make()
    h, L = dev(o["hash"].view(np.int32)), dev(o["lists"].view(np.int32))
    rs, _ = orc.bc_similarities(prox, bc, o["hash"], o["lists"], feats, stats)
    for steer in (False, True):
        room = torch.full((n * (K + 1) + 8,), -7.0, device="cuda")
        sims = room[4 + shift:4 + shift + n * (K + 1)]
        if steer:
            ctx.bc_similarities_steer(prox, sp, bc, h, L, dev(feats), dev(stats), empty_f32(n, 4), sims,
                                      dev(o["sorted_pos"]), dev(o["sorted_forward"]), dev(f0), empty_f32(n, 4))
        else:
            ctx.bc_similarities(prox, bc, h, L, dev(feats), dev(stats), empty_f32(n, 4), sims)
        assert same(sims.reshape(n, K + 1), rs)
        assert (room[:4 + shift] == -7.0).all() and (room[4 + shift + n * (K + 1):] == -7.0).all()
