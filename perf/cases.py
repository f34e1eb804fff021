"""The work that a user of this framework has it do, as cases to time and compare.

listed() covers the simulation step from the smallest flock (launches and
latency) to the largest configured one (4,194,304 agents with every option),
the batched step, the differentiable rollout in both directions, the
stage-by-stage plug-in calls, KNN lists, and the BehaviorClustering and list
consumer passes.  draw() gives more cases of the same ranges.

A pass of a step case starts again from the state that the program holds and
advances the flock `steps` steps, as an episode of a longer run does, so each
pass does the same work.
"""
from __future__ import annotations

import math

import numpy as np
import torch

CELL = 4.0
RADIUS = 4.0
DT = 0.05
WEIGHTS = (1.0, 0.8, 0.6)
MAX_SPEED = 1.0
MAX_FORCE = 0.5
FEATURE_RATE = 0.1
TARGET_WEIGHT = 0.5
WANDER_WEIGHT = 0.2
WANDER_SEED = 12345


def listed():
    return [
        # the smallest configured flock (4,096 boids, 25^3 cells, K 16): launches and latency
        {"name": "step_4k", "kind": "step", "n": 4096, "k": 16, "side": 100.0, "blobs": 0, "steps": 8},
        # an ordinary flock of odd size, about one agent per cell, every sorted copy kept
        {"name": "step_100k", "kind": "step", "n": 100003, "k": 32, "side": 186.0, "blobs": 0, "steps": 4,
         "sorted_sa": True},
        # the headline workload: 1,048,576 boids in 64 Gaussian blobs, K 32
        {"name": "step_blobs_1m", "kind": "step", "n": 1 << 20, "k": 32, "side": 400.0, "blobs": 64, "steps": 4},
        # the largest configured flock: 4,194,304 agents, K 64, targets, wander and the feature update
        {"name": "step_full_4m", "kind": "step", "n": 1 << 22, "k": 64, "side": 640.0, "blobs": 0, "steps": 2,
         "targets": True, "wander": True, "features": True},
        # 256 uneven flocks (1,024 to 65,536 agents, 0.5 agents per unit^3) advanced as one batch
        {"name": "batch_256", "kind": "batch", "flocks": 256, "lo": 1024, "hi": 65536, "sizes_seed": 0, "k": 32,
         "steps": 2},
        # a small differentiable rollout: final positions and the gradients of weights and state
        {"name": "rollout_4k", "kind": "rollout", "n": 4096, "k": 32, "side": 64.0, "steps": 20, "every": 10},
        # the configured differentiable flock (65,536 boids, checkpoints every 20)
        {"name": "rollout_65k", "kind": "rollout", "n": 65536, "k": 32, "side": 160.0, "steps": 100, "every": 20},
        # the plug-in layer's calls one by one (reorder, neighbourhoods, steering, features), odd size and K
        {"name": "staged_300k", "kind": "staged", "n": 300007, "k": 24, "side": 264.0, "blobs": 18},
        # nearest-neighbour lists (useKnn) at a crowded density
        {"name": "knn_200k", "kind": "knn", "n": 200003, "k": 16, "side": 148.0, "blobs": 0},
        # BehaviorClustering's steerForClustering: behaviour forces, adaptive similarities of
        # 8 features with the cluster steering, world-centre seek and integration
        {"name": "clustering_1m", "kind": "clustering", "n": 1 << 20, "k": 32, "side": 400.0, "blobs": 64,
         "features": 8},
        # cluster labels propagated over the lists (10 iterations, connector) and their hit rate
        {"name": "membership_1m", "kind": "membership", "n": 1 << 20, "k": 32, "side": 400.0, "blobs": 64,
         "iterations": 10},
        # the list consumers outside the step: slow to avoid, neighbourhood colour, move to a target
        {"name": "consumers_500k", "kind": "consumers", "n": 500009, "k": 32, "side": 312.0, "blobs": 31},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_world(rng, n):
    """A uniform flock of 0.25 to 32 agents per cell, or blobs as dense as the headline workload's."""
    if rng.random() < 0.5:
        per_cell = math.exp(rng.uniform(math.log(0.25), math.log(32.0)))
        cells = max(5, int(round((n / per_cell) ** (1.0 / 3.0))))
        return {"side": cells * CELL, "blobs": 0}
    cells = max(5, int(round(100.0 * (n / float(1 << 20)) ** (1.0 / 3.0))))
    return {"side": cells * CELL, "blobs": max(1, n // 16384)}


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "batch", "rollout", "staged", "knn", "clustering",
                       "membership", "consumers"])
    if kind == "batch":
        hi = _log_int(rng, 4096, 65536)
        return {"kind": kind, "flocks": rng.randint(3, 256), "lo": rng.randint(500, 2048), "hi": hi,
                "sizes_seed": rng.randrange(1 << 20), "k": rng.choice([16, 24, 32]), "steps": 2}
    if kind == "rollout":
        n = _log_int(rng, 1000, 65536)
        cells = max(5, int(round(n ** (1.0 / 3.0))))
        return {"kind": kind, "n": n, "k": rng.choice([16, 32]), "side": cells * CELL,
                "steps": rng.randint(5, 60), "every": rng.randint(4, 20)}
    n = _log_int(rng, 1000, {"step": 1 << 21, "knn": 1 << 18}.get(kind, 1 << 20))
    case = {"kind": kind, "n": n, **_draw_world(rng, n)}
    if kind == "step":
        case["k"] = rng.choice([16, 20, 32, 48, 64])
        case["steps"] = 2 if n > 300000 else 4
        for option in ("sorted_sa", "targets", "wander", "features"):
            if rng.random() < 0.3:
                case[option] = True
    elif kind == "knn":
        case["k"] = rng.choice([8, 16, 32])
    else:
        case["k"] = rng.choice([16, 24, 32, 48])
    if kind == "clustering":
        case["features"] = rng.choice([4, 6, 8, 16])
    if kind == "membership":
        case["iterations"] = 10
    return case


# ---------------------------------------------------------------- inputs

def _generator(seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _motion(g, n):
    """Headings uniform on the sphere with speeds in [0.5, 1], and a smoothed acceleration at rest."""
    d = torch.randn(n, 3, generator=g, device=g.device)
    d = d / d.norm(dim=1, keepdim=True).clamp_min(1e-6)
    speed = 0.5 + 0.5 * torch.rand(n, 1, generator=g, device=g.device)
    return torch.cat([d, speed], dim=1)


def _below(side):
    return float(np.nextafter(np.float32(side), np.float32(0)))


def _inputs(case, seed):
    """The flock's state by agent ID: pos, forward, smooth_accel as float4 rows."""
    g = _generator(seed)
    n, side = case["n"], case["side"]
    if case.get("blobs"):
        centres = torch.rand(case["blobs"], 3, generator=g, device=g.device) * side
        of = torch.randperm(n, generator=g, device=g.device) % case["blobs"]
        # folded back at the world's faces, so that no two agents share a corner
        xyz = side - (side - (centres[of] + 10.0 * torch.randn(n, 3, generator=g, device=g.device)).abs()).abs()
    else:
        xyz = torch.rand(n, 3, generator=g, device=g.device) * side
    xyz = xyz.clamp(0.0, _below(side))
    state = {"pos": torch.cat([xyz, torch.ones_like(xyz[:, :1])], dim=1), "forward": _motion(g, n)}
    state["smooth_accel"] = torch.zeros_like(state["pos"])
    if case["kind"] == "staged" or (case["kind"] == "step" and case.get("features")):
        state["features"] = torch.rand(n, 4, generator=g, device=g.device)
    if case.get("wander"):
        state["wander"] = 2.0 * torch.rand(n, 2, generator=g, device=g.device) - 1.0
    if case["kind"] == "clustering":
        state["vectors"] = torch.randn(n, case["features"], generator=g, device=g.device)
    if case["kind"] == "consumers":
        t = torch.rand(n, 3, generator=g, device=g.device) * side
        state["shape_targets"] = torch.cat([t, torch.ones_like(t[:, :1])], dim=1)
    return state


def _batch_sizes(case):
    g = np.random.Generator(np.random.PCG64(case["sizes_seed"]))
    return np.round(np.exp(g.uniform(math.log(case["lo"]), math.log(case["hi"]), case["flocks"]))).astype(np.int64)


def _batch_inputs(case, seed):
    """Flock f: sizes[f] agents uniform in a cube at 0.5 agents per unit^3, weights U[0.5, 1.5]."""
    g = _generator(seed)
    sizes = _batch_sizes(case)
    sides = (sizes / 0.5) ** (1.0 / 3.0)
    weights = (0.5 + torch.rand(len(sizes), 3, generator=g, device=g.device)).cpu().numpy().astype(np.float32)
    n = int(sizes.sum())
    side = torch.repeat_interleave(torch.tensor(sides, device=g.device, dtype=torch.float32),
                                   torch.tensor(sizes, device=g.device))
    xyz = torch.rand(n, 3, generator=g, device=g.device) * side[:, None]
    state = {"pos": torch.cat([xyz, torch.ones_like(xyz[:, :1])], dim=1), "forward": _motion(g, n)}
    state["smooth_accel"] = torch.zeros_like(state["pos"])
    return sizes, sides, weights, state


def _cells(side):
    return int(math.ceil(side / CELL))


def _targets(step, side):
    """Eight targets on tilted circular orbits around the world's centre."""
    t, out = step * DT, np.zeros((8, 3))
    for k in range(8):
        r, a, tilt = 60.0 + 15.0 * k, (0.1 + 0.02 * k) * t + 2.0 * math.pi * k / 8, math.pi * k / 8
        out[k] = (0.5 * side + r * math.cos(a), 0.5 * side + r * math.sin(a) * math.cos(tilt),
                  0.5 * side + r * math.sin(a) * math.sin(tilt))
    return out.astype(np.float32)


# ---------------------------------------------------------------- the program's set-up

class _State:
    pass


def prepare(case, seed):
    from behavert_amd.autograd import Rollout
    from behavert_amd.engine import Batch, Context, Flock
    from behavert_amd.types import BcParams, ProxParams, SteerParams
    from behavert_amd.workloads import cube_grid

    kind = case["kind"]
    s = _State()
    s.case = dict(case)
    s.ctx = Context(torch.cuda.current_device())
    prox = ProxParams.make(case["k"], RADIUS, use_knn=kind == "knn")
    steer = SteerParams.make(weights=WEIGHTS, radius=RADIUS, max_speed=MAX_SPEED, max_force=MAX_FORCE,
                             seek_world_center=kind == "clustering")

    def host(state):
        return {k: state[k].cpu().numpy() for k in ("pos", "forward", "smooth_accel")}

    if kind == "batch":
        sizes, sides, weights, state = _batch_inputs(case, seed)
        s.start = state
        s.flock = Batch(s.ctx, [cube_grid(float(x)) for x in sides], sizes, weights, prox, steer, host(state),
                        sorted_smooth_accel=False)
        return s
    grid = cube_grid(case["side"])
    s.grid, s.prox, s.steer = grid, prox, steer
    state = _inputs(case, seed)
    if kind == "rollout":
        s.start = state
        s.rollout = Rollout(s.ctx, grid, prox, steer, case["n"], DT, case["steps"], case["every"])
        s.weights = torch.tensor(WEIGHTS, device="cuda", requires_grad=True)
        s.leaves = [state[k].clone().requires_grad_(True) for k in ("pos", "forward", "smooth_accel")]
        # dL/d(final positions) of a quadratic loss toward points near the start
        s.goal = state["pos"][:, :3] + 0.5
        return s
    if case.get("wander"):
        steer.wander_weight = WANDER_WEIGHT
        steer.wander_seed = WANDER_SEED
    if case.get("targets"):
        steer.target_weight = TARGET_WEIGHT
        steer.set_targets(_targets(0, case["side"]))
    if kind in ("step", "staged"):
        s.start = state
        np_or_none = lambda k: state[k].cpu().numpy() if k in state else None  # noqa: E731
        s.flock = Flock(s.ctx, grid, prox, steer, host(state), features=np_or_none("features"),
                        wander=np_or_none("wander"), sorted_smooth_accel=bool(case.get("sorted_sa")))
        return s
    # passes over the sorted state and the lists that a step's first stages leave
    s.flock = Flock(s.ctx, grid, prox, steer, host(state))
    s.flock.reorder_sim_data()
    if kind == "knn":
        return s
    s.flock.compute_neighborhoods()
    n, k = case["n"], case["k"]
    f4 = lambda: torch.empty((n, 4), dtype=torch.float32, device="cuda")  # noqa: E731
    s.force = [f4(), f4(), f4()]
    if kind == "clustering":
        s.bc = BcParams.make(case["features"], adaptive=True, cluster_weight=0.9, alignment_weight=0.7)
        s.vectors = state["vectors"]
        s.stats = torch.tensor([1.0, 0.5, 0.0, 0.0], device="cuda").repeat(n, 1)
        s.stats_out = f4()
        s.sims = torch.empty((n, k + 1), dtype=torch.float32, device="cuda")
        s.out = [f4(), f4(), f4()]
    elif kind == "membership":
        s.member = [torch.zeros((n, 3), dtype=torch.float32, device="cuda") for _ in range(3)]
        s.connector = torch.empty((n, 2, 4), dtype=torch.float32, device="cuda")
    else:
        s.force[0].zero_()
        s.targets = state["shape_targets"]
        s.forward_out, s.color = f4(), f4()
    return s


def _restart(s):
    fl = s.flock
    fl.pos.copy_(s.start["pos"])
    fl.forward.copy_(s.start["forward"])
    fl.smooth_accel.copy_(s.start["smooth_accel"])
    if "features" in s.start:
        fl.features.copy_(s.start["features"])
    if "wander" in s.start:
        fl.wander.copy_(s.start["wander"])


def run(state):
    s, case = state, state.case
    kind = case["kind"]
    if kind == "rollout":
        from behavert_amd.autograd import rollout_final_pos

        final = rollout_final_pos(s.rollout, s.weights, *s.leaves)
        loss = 0.5 * ((final - s.goal) ** 2).sum()
        grads = torch.autograd.grad(loss, [s.weights, *s.leaves])
        return {"pos": final.detach(), "weights_grad": grads[0], "pos_grad": grads[1], "forward_grad": grads[2],
                "smooth_accel_grad": grads[3]}
    fl = s.flock
    if kind in ("step", "batch"):
        _restart(s)
        rate = FEATURE_RATE if case.get("features") else 0.0
        for i in range(case["steps"]):
            if case.get("targets"):
                fl.steer.set_targets(_targets(i, case["side"]))
            fl.step(DT, i, rate)
    elif kind == "staged":
        _restart(s)
        fl.reorder_sim_data()
        fl.compute_neighborhoods()
        fl.apply_steering(DT)
        fl.update_features(FEATURE_RATE)
    if kind in ("step", "batch", "staged"):
        out = {"pos": fl.pos, "forward": fl.forward, "smooth_accel": fl.smooth_accel,
               "sorted_pos": fl.sorted_pos, "sorted_forward": fl.sorted_forward, "hash": fl.hash,
               "cell_start": fl.cell_start, "cell_end": fl.cell_end, "lists": fl.lists}
        if kind == "staged" or case.get("sorted_sa"):
            out["sorted_smooth_accel"] = fl.sorted_smooth_accel
        if kind != "batch" and fl.features is not None:
            out["features"] = fl.features
        if case.get("wander"):
            out["wander"] = fl.wander
        return out
    ctx, prox = s.ctx, s.prox
    if kind == "knn":
        fl.compute_neighborhoods()
        return {"lists": fl.lists}
    if kind == "clustering":
        ctx.steer_forces(prox, s.steer, DT, 0, fl.sorted_pos, fl.sorted_forward, fl.hash, fl.lists, s.force[0])
        ctx.bc_similarities_steer(prox, s.steer, s.bc, fl.hash, fl.lists, s.vectors, s.stats, s.stats_out, s.sims,
                                  fl.sorted_pos, fl.sorted_forward, s.force[0], s.force[1])
        ctx.apply_steering_force(s.grid, s.steer, DT, fl.sorted_pos, fl.sorted_forward, fl.sorted_smooth_accel,
                                 fl.hash, s.force[1], *s.out, force_out=s.force[2])
        return {"similarities": s.sims, "stats": s.stats_out, "force": s.force[2], "pos": s.out[0],
                "forward": s.out[1], "smooth_accel": s.out[2]}
    if kind == "membership":
        ctx.cluster_membership(prox, case["iterations"], fl.hash, fl.lists, fl.sorted_pos, s.member[0], s.member[1],
                               connector=s.connector)
        ctx.cluster_hit_rate(prox, 1.5, fl.hash, fl.lists, fl.sorted_pos, s.member[1], s.member[2])
        return {"membership": s.member[1], "connector": s.connector, "hit_rate": s.member[2]}
    ctx.steer_and_slow_to_avoid_neighbors(prox, s.steer, fl.sorted_pos, fl.sorted_forward, fl.lists, s.forward_out,
                                          s.force[0], s.force[1])
    ctx.neighborhood_color(prox, (0.1, 0.2, 0.3), 1, fl.hash, fl.lists, s.color)
    ctx.move_towards_target(1, (0.0, 0.0, 0.0), fl.hash, fl.sorted_pos, s.targets, s.force[1], s.force[2])
    return {"forward": s.forward_out, "avoid": s.force[1], "color": s.color, "force": s.force[2]}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Bytes: each input of the pass read once and each output written once (per step where a pass
    is several); flops: the distance test of an average list's candidates and the sums over it."""
    kind, k = case["kind"], case["k"]
    stride = 4 * (k // 4 + 1)
    if kind == "batch":
        sizes = _batch_sizes(case)
        n = int(sizes.sum())
        cells = sum(_cells(float(x)) ** 3 for x in (sizes / 0.5) ** (1.0 / 3.0))
        density = 32.0
    else:
        n, cells = case["n"], _cells(case["side"]) ** 3
        density = n / cells
    found = min(float(k), 4.19 * density)  # entries of an average list
    # state in and out, sorted position and heading, hash pairs, lists, cell ranges
    step_bytes = n * (48 + 48 + 32 + 8 + 4 * stride) + 8 * cells
    step_flops = n * (8 * 6.4 * found + 40 * found + 150)
    if kind in ("step", "batch"):
        extra = n * (16 * bool(case.get("sorted_sa")) + 32 * bool(case.get("features")) + 16 * bool(case.get("wander")))
        return {"bytes": case["steps"] * (step_bytes + extra), "flops": case["steps"] * step_flops}
    if kind == "rollout":
        # a step of the forward direction, and one of its adjoint (the step's records in, gradients in and out)
        return {"bytes": case["steps"] * (step_bytes + n * (48 + 8 + 4 * stride + 96)),
                "flops": case["steps"] * n * (8 * 6.4 * found + 160 * found + 450)}
    if kind == "staged":
        return {"bytes": step_bytes + n * (16 + 32), "flops": step_flops}
    row = n * (4 + 4 * found)  # a list's count and entries
    if kind == "knn":
        return {"bytes": n * (16 + 4 * stride) + 8 * cells, "flops": n * 8 * 27 * density}
    if kind == "clustering":
        f = case["features"]
        return {"bytes": row + n * (8 + 48 + 4 * f + 32 + 4 * (k + 1) + 16 + 48),
                "flops": n * found * (40 + 2 * f + 40 + 40) + 200 * n}
    if kind == "membership":
        return {"bytes": row + n * (8 + 16 + 12 + 12 + 32 + 12), "flops": n * found * (case["iterations"] + 12)}
    return {"bytes": row + n * (8 + 32 + 16 + 16 + 16 + 16 + 16 + 16), "flops": n * (40 * found + 60)}


# ---------------------------------------------------------------- the same in 64 bits

def _key_cells(pos32, size):
    """Unclamped cell coordinates and the clamped key coordinates (below or above the grid: the far face)."""
    c = torch.floor(pos32 / CELL).to(torch.int64)
    top = size - 1
    return c, torch.where((c < 0) | (c > top), top, c)


def _neighbours(pos32, size, base, k):
    """Sorted order and the capped lists (x offset outermost, z innermost; the first k within the radius)
    of agents at pos32 (n, 3), float32: size (n, 1) grid cells per axis and base (n,) first key of each
    agent's grid.  The radius test is the float32 one, so the lists are those of any exact build."""
    n, dev = pos32.shape[0], pos32.device
    _, kc = _key_cells(pos32, size)
    gx = size[:, 0]
    key = base + (kc[:, 2] * gx + kc[:, 1]) * gx + kc[:, 0]
    skey, order = torch.sort(key, stable=True)
    sp = pos32[order]
    gx, base_s = gx[order], base[order]
    cells = int((base + gx.max() ** 3).max().item()) + 1 if n else 1
    counts = torch.zeros(cells, dtype=torch.int64, device=dev).index_add_(0, skey, torch.ones_like(skey))
    start = torch.cumsum(counts, 0) - counts
    cell = torch.floor(sp / CELL).to(torch.int64)
    lists = torch.full((n, k), -1, dtype=torch.int64, device=dev)
    found = torch.zeros(n, dtype=torch.int64, device=dev)
    me = torch.arange(n, device=dev)
    x, y, z = sp[:, 0], sp[:, 1], sp[:, 2]
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                q = cell + torch.tensor([dx, dy, dz], device=dev)
                ok = ((q >= 0) & (q < gx[:, None])).all(dim=1) & (found < k)
                at = torch.where(ok, base_s + (q[:, 2] * gx + q[:, 1]) * gx + q[:, 0], 0)
                live = torch.nonzero(ok & (counts[at] > 0))[:, 0]
                m = 0
                while live.numel():
                    j = start[at[live]] + m
                    rx, ry, rz = x[j] - x[live], y[j] - y[live], z[j] - z[live]
                    take = (torch.sqrt((rx * rx + ry * ry) + rz * rz) <= RADIUS) & (j != me[live])
                    i = live[take]
                    lists[i, found[i]] = j[take]
                    found[i] += 1
                    m += 1
                    live = live[(counts[at[live]] > m) & (found[live] < k)]
    width = max(1, int(found.max().item()))
    return order, lists[:, :width], found


def _safe_norm(v):
    """Length with a derivative of 0 at 0, and the unit vector (0 there)."""
    d2 = (v * v).sum(-1, keepdim=True)
    zero = d2 == 0
    length = torch.sqrt(torch.where(zero, 1.0, d2))
    return torch.where(zero, 0.0, length), torch.where(zero, 0.0, v / length)


def _truncate(v, most):
    length, unit = _safe_norm(v)
    return torch.where(length <= most, v, unit * most)


def _philox(step, ids):
    """The first two words of Philox4x32-10 with counter (step, 0, 0, 0) and key (seed, id)."""
    u = np.uint64
    low = u(0xFFFFFFFF)
    c = [np.full(len(ids), step, u), np.zeros(len(ids), u), np.zeros(len(ids), u), np.zeros(len(ids), u)]
    k0, k1 = u(WANDER_SEED), ids.astype(u)
    for r in range(10):
        if r:
            k0, k1 = (k0 + u(0x9E3779B9)) & low, (k1 + u(0xBB67AE85)) & low
        a, b = u(0xD2511F53) * c[0], u(0xCD9E8D57) * c[2]
        c = [(b >> u(32)) ^ c[1] ^ k0, b & low, (a >> u(32)) ^ c[3] ^ k1, a & low]
    return c[0], c[1]


def _flock_force(p, f, lists, found, weights):
    """Separation, alignment and cohesion over the lists, in sorted order; weights (n, 3) or (3,)."""
    hold = (lists >= 0)[..., None]
    j = lists.clamp_min(0)
    off = torch.where(hold, p[j] - p[:, None], 0.0)
    d2 = torch.where(hold, (off * off).sum(-1, keepdim=True), 1.0)
    some = (found > 0)[:, None]
    count = found.clamp_min(1)[:, None].to(p.dtype)
    sep = _safe_norm((-off / d2).sum(1) / count)[1]
    ali = torch.where(some, _safe_norm(torch.where(hold, f[j], 0.0).sum(1) / count - f)[1], 0.0)
    coh = _safe_norm(off.sum(1) / count)[1]
    w = weights if weights.dim() == 2 else weights[None]
    return sep * w[:, 0:1] + ali * w[:, 1:2] + coh * w[:, 2:3]


def _seek(p, f, s, target):
    return _truncate(target - p, MAX_SPEED) - f * s


def _integrate(p, f, s, a, force):
    slow = 0.2 * MAX_SPEED
    length, unit = _safe_norm(force)
    reach = (s / slow).clamp_max(1.0)
    cone = 1.0 - 2.0 * reach ** 20
    bend = (s <= slow) & (length > 0) & ((unit * f).sum(-1, keepdim=True) < cone)
    side = _safe_norm(force - f * (force * f).sum(-1, keepdim=True))[1]
    bent = (f * cone + side * torch.sqrt((1.0 - cone * cone).clamp_min(1e-300))) * length
    force = _truncate(torch.where(bend, bent, force), MAX_FORCE)
    a = a + (force - a) * min(max(9.0 * DT, 0.15), 0.4)
    v = _truncate(f * s + a * DT, MAX_SPEED)
    speed, unit = _safe_norm(v)
    return p + v * DT, unit, speed, a


def _steps64(case, state, size, base, weights, steps, wander=None):
    """`steps` steps in 64 bits from the float32 state, by agent ID; differentiable in its inputs."""
    p, f, s, a = state
    feat = case.get("feat64")
    n = p.shape[0]
    for i in range(steps):
        order, lists, found = _neighbours(p.detach()[:, :3].to(torch.float32), size, base, case["k"])
        sp, sf, ss, sa = p[order], f[order], s[order], a[order]
        w = weights[order] if weights.dim() == 2 else weights
        force = _flock_force(sp, sf, lists, found, w)
        if case.get("targets"):
            t = torch.tensor(_targets(i, case["side"]), dtype=torch.float64, device=p.device)
            force = force + TARGET_WEIGHT * _seek(sp, sf, ss, t[order % 8])
        if wander is not None:
            r = [torch.from_numpy((x >> np.uint64(8)).astype(np.float64)).to(p.device) / 16777216.0
                 for x in _philox(i, np.arange(n))]
            wander = (wander + (torch.stack(r, 1) * 2.0 - 1.0) * (12.0 * DT)).clamp(-1.0, 1.0)
            side = _safe_norm(torch.stack([-sf[:, 2], torch.zeros_like(sf[:, 0]), sf[:, 0]], 1))[1]
            up = torch.linalg.cross(side, sf)
            sw = wander[order]
            force = force + WANDER_WEIGHT * (side * sw[:, 0:1] + up * sw[:, 1:2])
        if feat is not None:
            own = feat[order]
            hold = (lists >= 0)[..., None]
            mean = torch.where(hold, own[lists.clamp_min(0)], 0.0).sum(1) / found.clamp_min(1)[:, None]
            new = torch.empty_like(feat)
            new[order] = torch.where((found > 0)[:, None], own + (mean - own) * FEATURE_RATE, own)
            feat = new
        np_, nf, ns, na = _integrate(sp, sf, ss, sa, force)
        back = torch.empty_like(order)
        back[order] = torch.arange(n, device=order.device)
        p, f, s, a = np_[back], nf[back], ns[back], na[back]
    return p, f, s, a, feat, wander


def _rows(p, f, s, a):
    return {"pos": torch.cat([p, torch.ones_like(s)], 1), "forward": torch.cat([f, s], 1),
            "smooth_accel": torch.cat([a, torch.zeros_like(s)], 1)}


def exact(case, seed):
    kind, k = case["kind"], case["k"]
    if kind == "knn":
        return None  # whole numbers only
    if kind == "rollout" and case["steps"] > 20:
        return None  # the trajectory's own sensitivity outgrows 32 bits
    if kind == "batch":
        sizes, sides, weights, state = _batch_inputs(case, seed)
        dev = state["pos"].device
        per = torch.tensor([_cells(float(x)) for x in sides], device=dev)
        of = torch.repeat_interleave(torch.arange(len(sizes), device=dev), torch.tensor(sizes, device=dev))
        size = per[of][:, None]
        base = (torch.cumsum(per ** 3, 0) - per ** 3)[of]
        w = torch.from_numpy(weights).to(dev).double()[of]
    else:
        state = _inputs(case, seed)
        dev, n = state["pos"].device, case["n"]
        size = torch.full((n, 1), _cells(case["side"]), dtype=torch.int64, device=dev)
        base = torch.zeros(n, dtype=torch.int64, device=dev)
        w = torch.tensor([float(np.float32(x)) for x in WEIGHTS], dtype=torch.float64, device=dev)
    start = (state["pos"][:, :3].double(), state["forward"][:, :3].double(), state["forward"][:, 3:].double(),
             state["smooth_accel"][:, :3].double())
    if kind in ("step", "batch", "staged"):
        held = dict(case, feat64=state["features"].double() if "features" in state else None)
        wander = state["wander"].double() if "wander" in state else None
        p, f, s, a, feat, wander = _steps64(held, start, size, base, w, case.get("steps", 1), wander)
        out = {**_rows(p, f, s, a), "sorted_pos": None, "sorted_forward": None, "hash": None, "cell_start": None,
               "cell_end": None, "lists": None}
        if feat is not None:
            out["features"] = feat
        if wander is not None:
            out["wander"] = wander
        return out
    if kind == "rollout":
        leaves = [w.clone().requires_grad_(True), *[x.clone().requires_grad_(True) for x in start]]
        p = _steps64(case, leaves[1:], size, base, leaves[0], case["steps"])[0]
        goal = (state["pos"][:, :3] + 0.5).double()
        g = torch.autograd.grad(0.5 * ((p - goal) ** 2).sum(), leaves)
        zero = torch.zeros_like(g[3])
        return {"pos": p.detach(), "weights_grad": g[0], "pos_grad": torch.cat([g[1], zero], 1),
                "forward_grad": torch.cat([g[2], g[3]], 1), "smooth_accel_grad": torch.cat([g[4], zero], 1)}
    order, lists, found = _neighbours(state["pos"][:, :3], size, base, k)
    p, f, s = (x[order] for x in start[:3])
    n = len(order)
    hold, j = lists >= 0, lists.clamp_min(0)
    some = (found > 0)[:, None]
    count = found.clamp_min(1)[:, None].double()

    def by_id(x):
        out = torch.empty_like(x)
        out[order] = x
        return out

    if kind == "membership":
        label = torch.arange(n, device=dev, dtype=torch.float64)
        for _ in range(case["iterations"]):
            label = torch.minimum(label, torch.where(hold, label[j], math.inf).min(1).values)
        sp = state["pos"].double()[order]
        close = hold & (torch.sqrt(((p[j] - p[:, None]) ** 2).sum(-1)) <= 1.5)
        m = close.sum(1)
        hit = (close & (label[j] == label[:, None])).sum(1) / m.clamp_min(1)
        mean = torch.where(m > 0, torch.where(close, label[j], 0.0).sum(1) / m.clamp_min(1), -1.0)
        zero = torch.zeros_like(label)
        return {"membership": by_id(torch.stack([label, zero, zero], 1)),
                "connector": by_id(torch.stack([sp, sp[label.long()]], 1)),
                "hit_rate": by_id(torch.stack([label, hit, mean], 1))}
    if kind == "consumers":
        off = torch.where(hold[..., None], p[j] - p[:, None], 0.0)
        d2 = torch.where(hold, (off * off).sum(-1), 1.0)[..., None]
        steering = _safe_norm((-off / d2).sum(1) / count)[1] * WEIGHTS[0]
        crowd = found[:, None].double()
        steering = torch.where(crowd > 16, steering * (crowd - 16.0) * 0.5, steering)
        c = (steering * f).sum(1, keepdim=True)
        speed = torch.where(c < -0.8, s * 0.9, torch.where(c > 0.5, s * 1.02, s))
        zero = torch.zeros_like(s)
        x = found.double() / k
        base_c = [float(np.float32(v)) for v in (0.1, 0.2, 0.3)]
        color = torch.stack([base_c[0] + x, base_c[1] + 0.3 + 1.0 - x, base_c[2] + x * (1.0 - x),
                             torch.ones_like(x)], 1)
        shifted = order + 1
        t = torch.cat([state["shape_targets"].double(), torch.zeros(1, 4, dtype=torch.float64, device=dev)])[shifted]
        pull = _safe_norm(t[:, :3] - p)[1] * 12.0 * t[:, 3:]
        return {"forward": torch.cat([f, speed], 1), "avoid": torch.cat([steering, zero], 1), "color": by_id(color),
                "force": torch.cat([pull + steering, zero], 1)}
    # clustering: the adaptive statistics follow the list, entry by entry
    vec = state["vectors"].double()[order]
    norm = vec.norm(dim=1)
    rate = [float(np.float32(v)) for v in (0.1, 0.1, 0.001)]
    mn, avg, mx = (torch.full((n,), v, dtype=torch.float64, device=dev) for v in (1.0, 0.5, 0.0))
    sims = torch.zeros(n, k + 1, dtype=torch.float64, device=dev)
    coh, ali = torch.zeros_like(p), torch.zeros_like(p)
    cw, aw = float(np.float32(0.9)), float(np.float32(0.7))
    for t in range(lists.shape[1]):
        live, o = hold[:, t], j[:, t]
        sim = ((vec * vec[o]).sum(1) / (norm * norm[o]) + 1.0) / 2.0
        navg = (avg + (sim - avg) * rate[0]).clamp(0.0, 1.0)
        lower = mn + (sim - mn) * rate[1]
        lower = torch.where(lower > navg, torch.minimum(lower, sim).clamp_min(0.0), lower)
        nmn = torch.where(sim < mn, lower, torch.where(mn < navg, mn + rate[2], mn))
        upper = mx + (sim - mx) * rate[1]
        upper = torch.where(upper < navg, torch.maximum(sim, upper.clamp_max(1.0)), upper)
        nmx = torch.where(sim > mx, upper, torch.where(mx > navg, mx - rate[2], mx))
        above = 0.5 * (sim - nmx) / (navg - nmx) + (sim - navg) / (nmx - navg)
        below = 0.5 * (sim - nmn) / (navg - nmn)
        out = torch.where(sim > navg, above, below).nan_to_num(0.0, 1.0, 0.0).clamp(0.0, 1.0)
        mn, avg, mx = (torch.where(live, x, y) for x, y in ((nmn, mn), (navg, avg), (nmx, mx)))
        out = torch.where(live, out, 0.0)
        sims[:, t] = out
        ahead = _truncate(p[o] - p, MAX_SPEED)
        both = (ahead - f * s) * out[:, None] + (-ahead - f * s) * (1.0 - out[:, None])
        coh = coh + torch.where(live[:, None], both, 0.0)
        ali = ali + torch.where(live[:, None], f[o] * out[:, None], 0.0)
    force = _flock_force(p, f, lists, found, w)
    force = force + torch.where(some, _safe_norm(coh / count)[1] * cw, 0.0)
    force = force + torch.where(some, _safe_norm(ali / count - f)[1] * aw, 0.0)
    half = 0.5 * _cells(case["side"]) * CELL
    inside = ((p - half).abs() < half - 2.0 * CELL).all(dim=1, keepdim=True)
    force = force + torch.where(inside, 0.0, _seek(p, f, s, torch.full_like(p, half)))
    zero = torch.zeros_like(s)
    stats = torch.stack([mn, avg, mx, torch.zeros_like(mn)], 1)
    new = _integrate(p, f, s, start[3][order], force)
    return {"similarities": sims, "stats": by_id(stats), "force": torch.cat([force, zero], 1),
            **{name: by_id(x) for name, x in _rows(*new).items()}}
