"""Launches of 3 x 2^20 agents and more with K beyond 32 map runs of workgroups to
the XCDs: a step with the feature update whose grid is no multiple of the runs'
256 workgroups has the same bits as one with the workgroups in order."""
import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.engine import Flock
from behavert_amd.types import OPT_XCD_REMAP, ProxParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(3 << 20) + 1, (3 << 20) + 12345])
def test_runs_with_a_remainder(ctx, n):
    side = 4.0 * 148
    g = torch.Generator(device="cuda").manual_seed(n)
    pos = torch.rand(n, 4, generator=g, device="cuda") * side
    fwd = torch.rand(n, 4, generator=g, device="cuda") - 0.5
    features = torch.rand(n, 4, generator=g, device="cuda")
    zero = np.zeros((n, 4), np.float32)
    state = {"pos": zero, "forward": zero, "smooth_accel": zero}
    out = []
    for remap in (0, 1):
        fl = Flock(ctx, W.cube_grid(side), ProxParams.make(33, 4.0), W.plain_steer(), state, features=zero)
        for a, b in ((fl.pos, pos), (fl.forward, fwd), (fl.features, features)):
            a.copy_(b)
        ctx.set_option(OPT_XCD_REMAP, remap)
        try:
            fl.step(0.05, 0, 0.1)
        finally:
            ctx.set_option(OPT_XCD_REMAP, 1)
        out.append([t.view(torch.int32) for t in (fl.lists, fl.pos, fl.forward, fl.smooth_accel, fl.features)])
    assert all(torch.equal(a, b) for a, b in zip(*out))
