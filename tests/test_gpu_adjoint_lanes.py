"""The adjoint with four lanes per agent (small flocks) and with one (large
ones) gives the same bits: the four lanes add their terms in list order.  The
same agents alone, and with others far above them (whose cotangents are zero)
that bring the flock to the largest size of the one and the smallest of the
other; list caps below, at and above what the four lanes hold at once, agents
outside the grid."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.types import GridParams, ProxParams

from ._adjoint_common import record_forward
from ._parity import f32
from .test_gpu_adjoint import adjoint_step

pytestmark = pytest.mark.gpu

QUAD_MAX = 1 << 17


@pytest.mark.parametrize("n,K", [(1, 4), (3, 1), (64, 8), (65, 9), (257, 32), (1500, 3), (1500, 20)])
def test_lanes_per_agent_give_the_same_bits(ctx, orc, n, K):
    rng = np.random.default_rng(n + K)
    side = 4.0 * max(3, round((n / 3.0) ** (1.0 / 3.0)))
    cells = int(side / 4.0)
    layers = max(60, 20000 // cells**2)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (cells, cells, cells + layers))
    steer = W.plain_steer((1.0, 0.8, 0.6))
    near = rng.uniform(-2.0, side, (n, 3))
    cot = [rng.standard_normal((n, 4)).astype(np.float32) for _ in range(3)]
    motion = W.directions_and_speeds(rng, QUAD_MAX + 1)
    got = []
    for total in (n, QUAD_MAX, QUAD_MAX + 1):
        far = np.random.default_rng(7).uniform([0.0, 0.0, side + 8.0], [side, side, side + 4.0 * (layers - 4)], (total - n, 3))
        st = W.make_state(np.concatenate([near, far]).astype(np.float32), *[m[:total] for m in motion])
        prox = ProxParams.make(K, 4.0)
        w = W.Workload("lanes", total, side, grid, prox, steer, 0.05, 1, st)
        _, recs = record_forward(orc, w, steer, 1)
        h, L, spos, sfwd = recs[0]
        ssa = st["smooth_accel"][h[:, 1].astype(np.int64)]
        g = [np.concatenate([c, np.zeros((total - n, 4), np.float32)]) for c in cot]
        wg = torch.zeros(3, dtype=torch.float32, device="cuda")
        gi = adjoint_step(ctx, grid, prox, steer, 0.05, spos, sfwd, ssa, h, L, *g, wg)
        got.append(([f32(x)[:n] for x in gi], f32(wg), L[:, 0].max()))
    assert n < 64 or K > 9 or got[0][2] == K
    for other in got[1:]:
        for a, b in zip(got[0][0], other[0]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        # the agents' weight terms, of magnitude <= 10 each, in another order of addition
        np.testing.assert_allclose(other[1], got[0][1], rtol=0, atol=10.0 * n * 2.0 ** -23)
