"""The scratch of a context against captures and other calls on the same context: a
step captured into a caller's graph after a warm-up with other options runs, a
captured step keeps its scratch while eager steps with other options run, and the
steps that move their state as records equal those that cannot; so for the passes
over the lists."""
import ctypes as C

import numpy as np
import pytest
import torch

from behavert_amd import workloads as W
from behavert_amd.autograd import Rollout
from behavert_amd.engine import Context, Flock, current_stream
from behavert_amd.types import OPT_STEP_GRAPH, ProxParams, SteerParams

pytestmark = pytest.mark.gpu

N, DT = 1 << 19, 0.05


@pytest.fixture
def own():
    """A context whose scratch no other test has grown."""
    c = Context(0)
    yield c
    torch.cuda.synchronize()
    c.close()


def inputs(K, n=N):
    side = 4.0 * round(n ** (1.0 / 3.0))
    return W.cube_grid(side), ProxParams.make(K, 4.0), W.uniform_flock(n, side, K)


def steer_with(wander):
    s = SteerParams.make(weights=(1.0, 0.8, 0.6))
    s.wander_weight = 0.3 if wander else 0.0
    return s


def flock(ctx, grid, prox, st, wander=False, features=False, sorted_sa=False):
    n = len(st["pos"])
    rng = np.random.default_rng(n)
    return Flock(ctx, grid, prox, steer_with(wander), st, sorted_smooth_accel=sorted_sa,
                 features=rng.uniform(0, 1, (n, 4)).astype(np.float32) if features else None,
                 wander=np.zeros((n, 2), np.float32))


def outputs(fl):
    names = ["pos", "forward", "smooth_accel", "lists", "hash", "wander"]
    return [getattr(fl, k).clone() for k in names] + ([fl.features.clone()] if fl.features is not None else [])


def same(a, b):
    return all(torch.equal(x.view(torch.int32), y.view(torch.int32)) for x, y in zip(a, b))


def eager(grid, prox, st, steps, **options):
    c = Context(0)
    fl = flock(c, grid, prox, st, **options)
    out = []
    for _ in range(steps):
        fl.step(DT, 0)
        out.append(outputs(fl))
    torch.cuda.synchronize()
    c.close()
    return out


def put(fl, st):
    for k in ("pos", "forward", "smooth_accel"):
        getattr(fl, k).copy_(torch.from_numpy(st[k]))
    fl.wander.zero_()


def capture(fl):
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        fl.step(DT, 0)
    return g


def replay_equals(g, fl, want):
    for w in want:
        g.replay()
        torch.cuda.synchronize()
        assert same(outputs(fl), w)


@pytest.mark.parametrize("wander,sorted_sa", [(True, False), (False, True), (True, True)])
def test_captured_after_a_warm_up_with_other_options(own, wander, sorted_sa):
    """Two-pass steps (K 100) whose records the warm-up did not need."""
    grid, prox, st = inputs(100)
    want = eager(grid, prox, st, 3, wander=wander, sorted_sa=sorted_sa)
    fl = flock(own, grid, prox, st)
    fl.step(DT, 0)
    fl.steer, fl.keep_sorted_smooth_accel = steer_with(wander), sorted_sa
    put(fl, st)
    replay_equals(capture(fl), fl, want)


def test_captured_step_keeps_its_scratch(own):
    """Eager steps with wander, features and the sorted copy between the replays of
    a step captured without them."""
    grid, prox, st = inputs(100)
    want = eager(grid, prox, st, 3)
    fl, other = flock(own, grid, prox, st), flock(own, grid, prox, st, wander=True, features=True, sorted_sa=True)
    fl.step(DT, 0)
    put(fl, st)
    g = capture(fl)
    other.step(DT, 0, 0.1)
    for w in want:
        g.replay()
        torch.cuda.synchronize()
        assert same(outputs(fl), w)
        other.step(DT, 1, 0.1)


@pytest.mark.parametrize("wander,features", [(True, False), (True, True)])
def test_step_graph_and_no_allocation_step(own, wander, features):
    """At the size of the records: brt_step's own graph, which has them, and the
    no-allocation step, which moves arrays, against direct launches."""
    grid, prox, st = inputs(64)
    flocks = [flock(own, grid, prox, st, wander=wander, features=features) for _ in range(3)]
    rate = 0.1 if features else 0.0
    for _ in range(5):
        flocks[0].step(DT, 0, rate)
        own.set_option(OPT_STEP_GRAPH, 1)
        flocks[1].step(DT, 0, rate)
        own.set_option(OPT_STEP_GRAPH, 0)
        fl, b = flocks[2], flocks[2].buffers()
        own.check(own._lib.brt_step_noalloc(own.handle, C.byref(grid), C.byref(prox), C.byref(fl.steer), rate, DT, 0,
                                            C.byref(b), current_stream()))
        if features:
            fl.features, fl.features_out = fl.features_out, fl.features
        torch.cuda.synchronize()
        assert same(outputs(flocks[0]), outputs(flocks[1])) and same(outputs(flocks[0]), outputs(flocks[2]))


@pytest.mark.parametrize("n,K", [((1 << 17) + 77, 48), (5000, 100)])
def test_captured_without_packed_positions(own, n, K):
    """Fused steps beyond K 32 after a warm-up whose search takes no packed
    positions: two passes with the feature update, KNN lists."""
    grid, prox, st = inputs(K, n)
    want = eager(grid, prox, st, 3)
    fl = flock(own, grid, prox, st, features=n > 1 << 17)
    if n > 1 << 17:
        fl.step(DT, 0, 0.1)
        fl.features = fl.features_out = None
    else:
        fl.prox = ProxParams.make(K, 4.0, use_knn=True)
        fl.step(DT, 0)
        fl.prox = prox
    put(fl, st)
    replay_equals(capture(fl), fl, want)


def test_hit_rate_captured_after_the_label_propagation(own):
    n = 20003
    grid, prox, st = inputs(16, n)
    other = Context(0)
    fl = flock(other, grid, prox, st)
    fl.reorder_sim_data()
    fl.compute_neighborhoods()
    zero = torch.zeros(n, 3, device="cuda")
    label, want, got = torch.empty_like(zero), torch.empty_like(zero), torch.empty_like(zero)
    own.cluster_membership(prox, 10, fl.hash, fl.lists, fl.sorted_pos, zero, label)
    other.cluster_hit_rate(prox, 3.0, fl.hash, fl.lists, fl.sorted_pos, label, want)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        own.cluster_hit_rate(prox, 3.0, fl.hash, fl.lists, fl.sorted_pos, label, got)
    for _ in range(3):
        got.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert same([got], [want])
    other.close()


def adjoint(c, n):
    """One step's records and adjoint seeds of a flock, ready for its adjoint call."""
    grid, prox, st = inputs(8, n)
    r = Rollout(c, grid, prox, steer_with(False), n, DT, 1, 1, overlap=False)
    r.forward((1.0, 0.8, 0.6), *[torch.from_numpy(st[k]).cuda() for k in ("pos", "forward", "smooth_accel")])
    r._replay(r.checkpoints[0], 0, c)
    for k, t in enumerate(r.g[0]):
        t.normal_(generator=torch.Generator(device="cuda").manual_seed(k))
    return r


def test_adjoint_captured_after_a_larger_flocks(own):
    """A flock of the four-lane adjoint, whose workgroups are smaller."""
    large, small, other = adjoint(own, 200003), adjoint(own, 131072), Context(0)
    large._adjoint(0, 0, 0)
    ref = adjoint(other, 131072)
    ref._adjoint(0, 0, 0)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        small._adjoint(0, 0, 0)
    for _ in range(3):
        small.wgrad.zero_()
        large._adjoint(0, 0, 0)
        g.replay()
        torch.cuda.synchronize()
        assert same([small.wgrad, *small.g[1]], [ref.wgrad, *ref.g[1]])
    other.close()
