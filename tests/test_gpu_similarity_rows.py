"""Where the similarity passes store their rows: 16 bytes per lane where the array
allows it, whole rows and partial ones, nothing outside them; alone and with the
cluster steering, on both sides of the sizes from which that pass reads its
neighbours as records, and without room for them.  Bit-exact against the CPU
oracle."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.engine import Context
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


def density_ramp(orc, n, K):
    """Agents of 1 to 60 per cell: the density rises along x."""
    rng = np.random.default_rng(K + n)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, (40, 30, 16))
    xyz = rng.uniform(0, 1, (n, 3)) ** (0.35, 1.0, 1.0) * (160.0, 120.0, 64.0)
    st = W.make_state(xyz.astype(np.float32), *W.directions_and_speeds(rng, n))
    prox = ProxParams.make(K, 4.0)
    return rng, prox, oracle_grid_outputs(orc, grid, prox, st)


def inputs(orc, n, K, F, adaptive):
    rng, prox, o = density_ramp(orc, n, K)
    feats = (rng.standard_normal((n, F)) + rng.standard_normal(F)).astype(np.float32)
    stats = np.sort(rng.uniform(0, 1, (n, 4)), axis=1).astype(np.float32)
    f0 = rng.standard_normal((n, 4)).astype(np.float32)
    bc, sp = BcParams.make(F, adaptive=adaptive), SteerParams.make()
    rs, rst = orc.bc_similarities(prox, bc, o["hash"], o["lists"], feats, stats if adaptive else None)
    rf = orc.bc_cluster_steer(prox, sp, bc, o["sorted_pos"], o["sorted_forward"], o["lists"], rs, f0)
    args = [dev(a) for a in (o["hash"].view(np.int32), o["lists"].view(np.int32), feats, stats)]
    return prox, bc, sp, args, [dev(o["sorted_pos"]), dev(o["sorted_forward"]), dev(f0)], (rs, rst, rf)


LEAST, WIDE = 9 << 14, 3 << 16


@pytest.mark.parametrize("n,K,F,adaptive", [(LEAST - 1, 32, 8, True), (LEAST, 32, 8, True), (LEAST + 63, 3, 5, False),
                                            (LEAST + 1, 35, 9, True), (LEAST + 1, 36, 25, True),
                                            (LEAST + 63, 48, 24, False), (LEAST, 49, 16, True),
                                            (WIDE + 1, 24, 4, True), (WIDE + 63, 48, 1, False), (WIDE - 1, 32, 4, True),
                                            (WIDE + 1, 64, 8, True), (WIDE + 63, 80, 32, True), (WIDE, 81, 12, True)])
def test_records(ctx, orc, n, K, F, adaptive):
    prox, bc, sp, args, state, (rs, rst, rf) = inputs(orc, n, K, F, adaptive)
    sims = torch.full((n, K + 1), float("nan"), device="cuda")
    st, out = empty_f32(n, 4), empty_f32(n, 4)
    ctx.bc_similarities_steer(prox, sp, bc, *args, st, sims, *state, out)
    assert same(sims, rs) and same(out, rf)
    if adaptive:
        assert same(st, rst)


SOON = 3 << 15


@pytest.mark.parametrize("n,K,F,adaptive", [(SOON - 1, 32, 8, True), (SOON, 32, 8, True), (SOON + 63, 24, 5, False),
                                            (SOON, 23, 8, True), (SOON + 1, 36, 6, True), (SOON + 1, 4, 9, True),
                                            (SOON, 48, 16, True), (LEAST + 1, 16, 8, True), (WIDE - 1, 16, 4, True),
                                            (WIDE + 63, 16, 3, False), (WIDE, 15, 4, True)])
def test_records_by_list_and_feature_length(ctx, orc, n, K, F, adaptive):
    test_records(ctx, orc, n, K, F, adaptive)


def test_captured_without_room_for_records(orc):
    """A warm-up with the similarities alone, then the pass with the steering captured."""
    n, K, F = LEAST + 5, 32, 8
    prox, bc, sp, args, state, (rs, rst, rf) = inputs(orc, n, K, F, True)
    own = Context(0)
    sims, st, out = torch.empty((n, K + 1), device="cuda"), empty_f32(n, 4), empty_f32(n, 4)
    own.bc_similarities(prox, bc, *args, st, sims)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        own.bc_similarities_steer(prox, sp, bc, *args, st, sims, *state, out)
    for _ in range(3):
        for t in (sims, st, out):
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert same(sims, rs) and same(st, rst) and same(out, rf)
    own.close()


@pytest.mark.parametrize("n,steer", [(SOON + 63, False), (SOON - 1, True), (1000, False)])
def test_captured_after_a_pass_from_records(orc, n, steer):
    """A warm-up from records, then the similarities alone, or a flock too small for
    records, captured: the call has the scratch it needs."""
    K, F = 32, 8
    own = Context(0)
    prox, bc, sp, args, state, _ = inputs(orc, SOON + 63, K, F, True)
    own.bc_similarities_steer(prox, sp, bc, *args, empty_f32(SOON + 63, 4), torch.empty((SOON + 63, K + 1), device="cuda"),
                              *state, empty_f32(SOON + 63, 4))
    prox, bc, sp, args, state, (rs, rst, rf) = inputs(orc, n, K, F, True)
    sims, st, out = torch.empty((n, K + 1), device="cuda"), empty_f32(n, 4), empty_f32(n, 4)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        if steer:
            own.bc_similarities_steer(prox, sp, bc, *args, st, sims, *state, out)
        else:
            own.bc_similarities(prox, bc, *args, st, sims)
    for _ in range(3):
        for t in (sims, st, out):
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert same(sims, rs) and same(st, rst) and (not steer or same(out, rf))
    own.close()
