"""GPU parity of the passes over the lists on both sides of the launch size from
which their waves load the rows together (73,728 agents): row widths at which the
loading changes (K 3, 16, 32 and 35 staged whole, from 36 on in blocks), lists
that end in each block, a last wave of one agent and of 63.  Bit-exact against
the CPU oracle."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.types import BcParams, GridParams, ProxParams, SteerParams

from ._parity import dev, empty_f32, f32, first_mismatch, oracle_grid_outputs

pytestmark = pytest.mark.gpu

OWN = 73728  # the largest launch whose lanes read their own rows


def flock(orc, n, K):
    """Agents of 1 to 60 per cell: the density rises along x."""
    rng = np.random.default_rng(K + n)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (30, 24, 12))
    xyz = rng.uniform(0, 1, (n, 3)) ** (0.35, 1.0, 1.0) * (120.0, 96.0, 48.0)
    st = W.make_state(xyz.astype(np.float32), *W.directions_and_speeds(rng, n))
    prox = ProxParams.make(K, 4.0)
    return rng, grid, prox, oracle_grid_outputs(orc, grid, prox, st)


def same(a, b):
    return first_mismatch(f32(a).view(np.uint32), np.ascontiguousarray(b, np.float32).view(np.uint32)) is None


@pytest.mark.parametrize("n,K", [(OWN, 35), (OWN, 36), (OWN + 1, 3), (OWN + 1, 16), (OWN + 1, 32), (OWN + 63, 35),
                                 (OWN + 1, 36), (OWN + 63, 48), (OWN + 63, 63), (OWN + 1, 100), (OWN + 63, 252)])
def test_passes(ctx, orc, n, K):
    rng, grid, prox, o = flock(orc, n, K)
    h, L = dev(o["hash"].view(np.int32)), dev(o["lists"].view(np.int32))
    pos, fwd, ssa = dev(o["sorted_pos"]), dev(o["sorted_forward"]), dev(o["sorted_smooth_accel"])
    fin = rng.standard_normal((n, 4)).astype(np.float32)
    sp = SteerParams.make(weights=(1.3, 0.8, 0.6), radius=3.0, cos_max=-0.5, min_radius=0.5)
    out = [empty_f32(n, 4) for _ in range(3)]
    ctx.steer_forces(prox, sp, 0.05, 0, pos, fwd, h, L, out[0])
    rforce, _ = orc.steer_forces(prox, sp, 0.05, 0, o["sorted_pos"], o["sorted_forward"], o["hash"], o["lists"])
    assert same(out[0], rforce)
    ctx.steer_integrate(grid, prox, sp, 0.05, 0, pos, fwd, ssa, h, L, *out)
    want = orc.steer_f32(grid, prox, sp, 0.05, 0, o["sorted_pos"], o["sorted_forward"], o["sorted_smooth_accel"],
                         o["hash"], o["lists"])
    assert all(same(a, b) for a, b in zip(out, (want[k] for k in ("pos", "forward", "smooth_accel"))))
    ctx.feature_update(prox, 0.1, h, L, dev(fin), out[0])
    assert same(out[0], orc.feature_update_f32(prox, 0.1, o["hash"], o["lists"], fin))
    m = [torch.zeros((n, 3), dtype=torch.float32, device="cuda") for _ in range(2)]
    conn = empty_f32(n, 2, 4)
    for iterations in (1, 3):
        ctx.cluster_membership(prox, iterations, h, L, pos, m[0], m[1], connector=conn)
        rm, rc = orc.cluster_membership(prox, iterations, o["hash"], o["lists"], o["sorted_pos"], connector=True)
        assert same(m[1], rm) and same(conn, rc)
    bc, sims = BcParams.make(4), rng.uniform(0, 1, (n, K + 1)).astype(np.float32)
    ctx.bc_steer_for_clustering(prox, sp, bc, pos, fwd, L, dev(sims), dev(fin), out[1])
    assert same(out[1], orc.bc_cluster_steer(prox, sp, bc, o["sorted_pos"], o["sorted_forward"], o["lists"], sims, fin))
