"""GPU parity of the passes whose waves load their list rows together: every
row width at which the staging changes (K 3, 32 and 35: rows staged whole; 36
and more: blocks of 32 words; 238 and 239: the one-pass similarities + cluster
steering on both sides of its LDS limit), lists that end at a block's edge,
flocks that end inside a wave, features around the record's rounds.  Bit-exact
against the CPU oracle."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.types import BcParams, GridParams, ProxParams, SteerParams

from ._parity import dev, empty_f32, f32, first_mismatch, oracle_grid_outputs

pytestmark = pytest.mark.gpu


def flock(orc, n, K, seed):
    """A third of the agents crowded in one corner: short lists and full ones."""
    rng = np.random.default_rng(seed)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (6,) * 3)
    xyz = rng.uniform(0, 24, (n, 3))
    xyz[::3] *= 0.25
    st = W.make_state(xyz.astype(np.float32), *W.directions_and_speeds(rng, n))
    prox = ProxParams.make(K, 4.0)
    return rng, prox, oracle_grid_outputs(orc, grid, prox, st)


def same(a, b):
    return first_mismatch(f32(a).view(np.uint32), np.ascontiguousarray(b, np.float32).view(np.uint32)) is None


@pytest.mark.parametrize("K", [3, 16, 31, 32, 35, 36, 63, 64, 100, 252])
@pytest.mark.parametrize("n", [1, 63, 65, 2000])
def test_list_walks(ctx, orc, K, n):
    rng, prox, o = flock(orc, n, K, 7 * K + n)
    h, L = dev(o["hash"].view(np.int32)), dev(o["lists"].view(np.int32))
    pos, fwd = dev(o["sorted_pos"]), dev(o["sorted_forward"])
    fin = rng.standard_normal((n, 4)).astype(np.float32)
    sp = SteerParams.make(weights=(1.3, 0.8, 0.6), radius=3.0, cos_max=-0.5, min_radius=0.5)
    sp.alignment[1] = 2.5  # the separation's own radius decides in the slow-to-avoid pass
    out, out2 = empty_f32(n, 4), empty_f32(n, 4)
    ctx.steer_forces(prox, sp, 0.05, 0, pos, fwd, h, L, out)
    rforce, _ = orc.steer_forces(prox, sp, 0.05, 0, o["sorted_pos"], o["sorted_forward"], o["hash"], o["lists"])
    assert same(out, rforce)
    ctx.steer_and_slow_to_avoid_neighbors(prox, sp, pos, fwd, L, out2, dev(fin), out)
    rf, rforce = orc.slow_avoid(prox, sp, o["sorted_pos"], o["sorted_forward"], o["lists"], fin)
    assert same(out2, rf) and same(out, rforce)
    ctx.feature_update(prox, 0.1, h, L, dev(fin), out)
    assert same(out, orc.feature_update_f32(prox, 0.1, o["hash"], o["lists"], fin))
    m = [torch.zeros((n, 3), dtype=torch.float32, device="cuda") for _ in range(3)]
    conn = empty_f32(n, 2, 4)
    ctx.cluster_membership(prox, 3, h, L, pos, m[0], m[1], connector=conn)
    rm, rc = orc.cluster_membership(prox, 3, o["hash"], o["lists"], o["sorted_pos"], connector=True)
    assert same(m[1], rm) and same(conn, rc)
    ctx.cluster_hit_rate(prox, 1.5, h, L, pos, m[1], m[2])
    assert same(m[2], orc.cluster_hit_rate(prox, 1.5, o["hash"], o["lists"], o["sorted_pos"], rm))


@pytest.mark.parametrize("K,F", [(3, 1), (32, 8), (32, 9), (35, 4), (36, 8), (48, 24), (64, 25), (238, 5), (239, 5),
                                 (252, 32)])
@pytest.mark.parametrize("n", [1, 65, 1500])
@pytest.mark.parametrize("adaptive", [False, True])
def test_similarities_and_cluster_steering(ctx, orc, K, F, n, adaptive):
    rng, prox, o = flock(orc, n, K, 11 * K + n)
    feats = (rng.standard_normal((n, F)) + rng.standard_normal(F)).astype(np.float32)
    stats = np.zeros((n, 4), np.float32)
    stats[:, :3] = np.sort(rng.uniform(0, 1, (n, 3)), axis=1)
    bc, sp = BcParams.make(F, adaptive=adaptive), SteerParams.make()
    f0 = rng.standard_normal((n, 4)).astype(np.float32)
    sims = torch.full((n, K + 1), float("nan"), dtype=torch.float32, device="cuda")
    st, out = empty_f32(n, 4), empty_f32(n, 4)
    ctx.bc_similarities_steer(prox, sp, bc, dev(o["hash"].view(np.int32)), dev(o["lists"].view(np.int32)), dev(feats),
                              dev(stats), st, sims, dev(o["sorted_pos"]), dev(o["sorted_forward"]), dev(f0), out)
    rs, rst = orc.bc_similarities(prox, bc, o["hash"], o["lists"], feats, stats if adaptive else None)
    assert same(sims, rs)
    if adaptive:
        assert same(st, rst)
    assert same(out, orc.bc_cluster_steer(prox, sp, bc, o["sorted_pos"], o["sorted_forward"], o["lists"], rs, f0))
