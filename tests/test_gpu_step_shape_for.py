"""The reported launch shape of a step is the one that the step takes: whether the
steering ran as a pass of its own is read from the per-phase times, at sizes, K, grids
and with features on both sides of every rule; and the expected shapes themselves."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.engine import Flock
from behavert_amd.types import GridParams, OPT_FUSED_STEP, OPT_LDS_LISTS, ProxParams

pytestmark = pytest.mark.gpu

BIG = 1 << 21
SPARSE, CROWDED = (144, 128, 128), (64, 64, 64)

CASES = [
    # n, K, cells, features, (fused, LDS lists, lanes per agent)
    (1000, 16, CROWDED, False, (True, True, 4)),
    (1 << 17, 16, CROWDED, False, (True, True, 4)),
    ((1 << 17) + 1, 16, CROWDED, False, (True, True, 1)),
    (1000, 64, CROWDED, False, (True, True, 4)),
    (1000, 64, CROWDED, True, (False, True, 4)),
    (200000, 32, CROWDED, True, (True, True, 1)),
    (200000, 33, CROWDED, False, (True, True, 1)),
    (200000, 33, CROWDED, True, (False, False, 1)),
    (200000, 80, SPARSE, False, (True, True, 1)),
    (200000, 81, SPARSE, False, (False, False, 1)),
    (BIG - 1, 64, SPARSE, False, (True, True, 1)),
    (BIG, 64, SPARSE, False, (False, False, 1)),
    (BIG, 64, CROWDED, False, (True, True, 1)),
    (BIG, 64, CROWDED, True, (False, True, 1)),
    (BIG - 1, 64, CROWDED, True, (False, False, 1)),
]


@pytest.fixture
def automatic(ctx):
    old = ctx.get_option(OPT_FUSED_STEP), ctx.get_option(OPT_LDS_LISTS)
    ctx.set_option(OPT_FUSED_STEP, -1)
    ctx.set_option(OPT_LDS_LISTS, -1)
    yield ctx
    ctx.set_option(OPT_FUSED_STEP, old[0])
    ctx.set_option(OPT_LDS_LISTS, old[1])


def steers_apart(ctx, n, K, size, features, use_knn=False):
    rng = np.random.default_rng(1)
    grid = GridParams.direct((0.0,) * 3, (4.0,) * 3, size)
    st = W.make_state((rng.random((n, 3), np.float32) * (4.0 * np.array(size, np.float32))).astype(np.float32),
                      *W.directions_and_speeds(rng, n))
    fl = Flock(ctx, grid, ProxParams.make(K, 1.0, use_knn=use_knn), W.plain_steer(), st,
               features=rng.random((n, 4), np.float32) if features else None)
    ctx.phase_timing(True)
    fl.step(0.05, 0, 0.1 if features else 0.0)
    torch.cuda.synchronize()
    ms, steps = ctx.phase_times()
    ctx.phase_timing(False)
    assert steps == 1
    return ms["steer_integrate"] > 0.0


@pytest.mark.parametrize("n,K,size,features,want", CASES)
def test_the_step_takes_the_reported_shape(automatic, n, K, size, features, want):
    got = automatic.step_shape_for(ProxParams.make(K, 1.0), n, int(np.prod(size)), features)
    assert got == want
    assert steers_apart(automatic, n, K, size, features) == (not got[0])


def test_options_and_knn(automatic):
    ctx = automatic
    cells = int(np.prod(CROWDED))
    assert ctx.step_shape_for(ProxParams.make(16, 4.0, use_knn=True), 1000, cells) == (False, True, 1)
    assert steers_apart(ctx, 1000, 16, CROWDED, False, use_knn=True)
    ctx.set_option(OPT_FUSED_STEP, 0)
    assert ctx.step_shape_for(ProxParams.make(16, 4.0), 1 << 18, cells) == (False, True, 1)
    ctx.set_option(OPT_LDS_LISTS, 0)
    assert ctx.step_shape_for(ProxParams.make(16, 4.0), 1000, cells) == (False, False, 1)
    ctx.set_option(OPT_FUSED_STEP, 1)
    assert ctx.step_shape_for(ProxParams.make(64, 4.0), 1 << 18, cells) == (True, False, 1)
