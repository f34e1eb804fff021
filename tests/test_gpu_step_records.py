"""Steps that move the state by ID as records (two passes, 2^19 agents or more,
with features, wander or the sorted smoothed acceleration) and those on the other
side of each rule: bit-exact against the CPU oracle."""
import numpy as np
import pytest

from behavert_amd import workloads as W
from behavert_amd.engine import Flock
from behavert_amd.types import OPT_FUSED_STEP, ProxParams, SteerParams

from ._parity import first_mismatch, u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K,options", [((1 << 19) - 1, 64, "features wander"), (1 << 19, 64, "features wander"),
                                         ((1 << 19) + 3, 36, "features"), ((1 << 19) + 61, 48, "wander"),
                                         (1 << 19, 40, "sorted_sa"), ((1 << 19) + 1, 33, ""),
                                         ((1 << 19) + 2, 16, "features sorted_sa two_pass")])
def test_step_on_both_sides(ctx, orc, n, K, options):
    side = 4.0 * round(n ** (1.0 / 3.0))
    st = W.uniform_flock(n, side, n)
    rng = np.random.default_rng(K)
    st["smooth_accel"] = rng.uniform(-0.1, 0.1, (n, 4)).astype(np.float32)  # a fourth component to keep
    features = rng.uniform(0, 1, (n, 4)).astype(np.float32) if "features" in options else None
    wander = rng.uniform(-1, 1, (n, 2)).astype(np.float32) if "wander" in options else None
    steer = SteerParams.make(weights=(1.0, 0.8, 0.6), targets=W.moving_targets(0.3, 12.0), target_weight=0.4)
    steer.wander_weight = 0.3 if "wander" in options else 0.0
    grid, prox = W.cube_grid(side), ProxParams.make(K, 4.0)
    rate = 0.1 if features is not None else 0.0
    if "two_pass" in options:
        ctx.set_option(OPT_FUSED_STEP, 0)
    try:
        fl = Flock(ctx, grid, prox, steer, st, features=features, wander=wander,
                   sorted_smooth_accel="sorted_sa" in options)
        hf = orc.HostFlock(grid, prox, st, features=features, wander=wander)
        for step in range(2):
            fl.step(0.05, step, rate)
            hf.step(steer, 0.05, step, rate)
    finally:
        ctx.set_option(OPT_FUSED_STEP, -1)
    assert first_mismatch(u32(fl.lists), hf.lists) is None
    got = fl.state()
    for k in ("pos", "forward", "smooth_accel"):
        assert first_mismatch(got[k].view(np.uint32), getattr(hf, k).view(np.uint32)) is None, k
    if features is not None:
        assert first_mismatch(u32(fl.features), hf.features.view(np.uint32)) is None
    if wander is not None:
        assert first_mismatch(u32(fl.wander), hf.wander.view(np.uint32)) is None
