"""The work a user of this engine has it do, as measurable cases.

A case is one pass through the public entry points: place the agents, run
schedule steps, read the result.  Sizes are those of the flockers
configurations this repository runs elsewhere (1,000 boids on 200 x 200,
1,048,576 on 20,480 x 20,480, 8,388,608 in Gaussian blobs, ensembles of
1,000 to 262,144 agents) and what lies between them.

Every pass starts a run again from its initial state, so a pass is the same
work however often it is repeated.
"""
import ctypes
import math

import numpy as np
import torch

from krabmaga_amd import Ensemble, Field2D, FlockParams, RunSpec, _abi, lib, serve, workloads

D = 10.0 / 1.5    # discretization of the flockers configurations
RADIUS = 10.0     # Bird::step's neighbour radius
DENSE = 0.025     # birds per unit^2 of 1,000 boids on 200 x 200
SPARSE = 0.0025   # of 1,048,576 boids on 20,480 x 20,480
STATE = ("id", "x", "y", "hx", "hy")


def listed():
    return [
        # a visualiser's loop: one schedule step, the birds read and drawn,
        # the next step.  The smallest call: launches and latency count.
        {"name": "viewer 1000", "kind": "frames", "agents": 1000, "side": 200.0, "steps": 20},
        # the plain 1,000-boid configuration
        {"name": "field 1000", "kind": "field", "agents": 1000, "side": 200.0, "steps": 200},
        # ordinary single simulations at the same density, up to where a
        # field fills the chip
        {"name": "field 16384", "kind": "field", "agents": 16384, "side": 809.5, "steps": 200},
        {"name": "field 65537", "kind": "field", "agents": 65537, "side": 1619.1, "steps": 200},
        {"name": "field 262144", "kind": "field", "agents": 262144, "side": 3238.2,
         "steps": 200},
        # the headline configuration: a sparse million-boid field, 1,000 steps
        {"name": "field 1M sparse", "kind": "field", "agents": 1 << 20, "side": 20480.0,
         "steps": 1000},
        # clustered density: agents the caller places, crowded blobs on a
        # sparse background
        {"name": "blobs 8M", "kind": "blobs", "agents": 1 << 23, "side": 40960.0, "blobs": 64,
         "steps": 100},
        # exploration: a sweep of small runs, and replicas of uneven size
        {"name": "sweep of small runs", "kind": "ensemble", "replicas": 256, "n_min": 1000,
         "n_max": 4000, "steps": 200},
        {"name": "uneven replicas", "kind": "ensemble", "replicas": 96, "n_min": 1000,
         "n_max": 262144, "steps": 300},
        # serving: a queue of runs of different lengths, admitted together,
        # each read and retired when it is done
        {"name": "serve 32 runs", "kind": "serve", "replicas": 32, "n_min": 1000,
         "n_max": 262144, "s_min": 50, "s_max": 400},
        # every agent's neighbour vector (analysis of a field between steps)
        {"name": "neighbours 300001", "kind": "neighbours", "agents": 300001, "side": 3464.1},
        # one step over arrays that the caller keeps on the device
        {"name": "static step 500001", "kind": "static", "agents": 500001, "side": 4472.1},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _density(case):
    return case["agents"] / case["side"] ** 2


def _side(rng, n):
    """A torus for n agents at a density between the two configurations'."""
    return round(math.sqrt(n / _log(rng, SPARSE, DENSE)), 1)


def draw(rng):
    kind = rng.choice(["frames", "field", "field", "field", "field", "blobs", "ensemble",
                       "ensemble", "serve", "neighbours", "static"])
    c = {"kind": kind, "weights": rng.randrange(1 << 20)}
    if kind == "frames":
        n = int(_log(rng, 500, 20000))
        c.update(agents=n, side=_side(rng, n), steps=rng.randint(5, 30))
    elif kind == "field":
        n = int(_log(rng, 500, 1 << 20))
        steps = int(_log(rng, 20, 1000))
        c.update(agents=n, side=_side(rng, n), steps=min(steps, int(2e8 / n) + 20))
    elif kind == "blobs":
        n = int(_log(rng, 1 << 18, 1 << 22))
        blobs = max(1, n >> 17)
        c.update(agents=n, side=round(math.sqrt(n / 0.005), 1), blobs=blobs,
                 steps=rng.randint(10, 60))
    elif kind == "ensemble":
        top = int(_log(rng, 1500, 200000))
        c.update(replicas=max(4, min(300, int(1.5e6 / top))), n_min=500, n_max=top,
                 steps=rng.randint(20, 200))
    elif kind == "serve":
        top = int(_log(rng, 3000, 200000))
        c.update(replicas=rng.randint(8, 32), n_min=500, n_max=top, s_min=20,
                 s_max=rng.randint(60, 300))
    else:
        n = int(_log(rng, 1000, 600000))
        c.update(agents=n, side=_side(rng, n))
    return c


def _params(case, seed):
    """All weights 1 and jump 0.7 as configured, or a sampled vector as the
    exploration sweeps draw it."""
    if "weights" not in case:
        return FlockParams(radius=RADIUS, seed=seed)
    w = np.random.default_rng(case["weights"])
    v = [float(t) for t in w.uniform(0.5, 2.0, size=5)]
    return FlockParams(cohesion=v[0], avoidance=v[1], consistency=v[2], randomness=v[3],
                       momentum=v[4], jump=float(w.uniform(0.3, 1.0)), radius=RADIUS, seed=seed)


def _sizes(case):
    """Run sizes of an ensemble: log-uniform, the same for every seed."""
    g = np.random.default_rng(case.get("weights", 3))
    lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
    n = [int(math.exp(g.uniform(lo, hi))) for _ in range(case["replicas"])]
    steps = [int(s) for s in g.integers(case.get("s_min", 1), case.get("s_max", 1) + 1,
                                        size=len(n))]
    return n, steps


def _specs(case, seed):
    g = np.random.default_rng(seed)
    specs = []
    for i, n in enumerate(_sizes(case)[0]):
        w = [float(t) for t in g.uniform(0.5, 2.0, size=5)]
        side = math.sqrt(n / DENSE)
        key = (seed << 20) | i
        p = FlockParams(cohesion=w[0], avoidance=w[1], consistency=w[2], randomness=w[3],
                        momentum=w[4], jump=float(g.uniform(0.3, 1.0)), radius=RADIUS, seed=key)
        specs.append(RunSpec(width=side, height=side, agents=n, params=p, discretization=D,
                             heading_mode=1, init_seed=key))
    return specs


def _result(n):
    """Where a program collects the birds of many runs."""
    return {k: np.zeros(n, np.float32) for k in STATE[1:]}


def _static_inputs(case, seed):
    """Agents in random order, uniform positions, unit headings."""
    n, side = case["agents"], case["side"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    ids = torch.randperm(n, generator=g, device="cuda").to(torch.int32)
    x = torch.rand(n, generator=g, device="cuda") * side
    y = torch.rand(n, generator=g, device="cuda") * side
    a = torch.rand(n, generator=g, device="cuda") * (2.0 * math.pi)
    return ids, x, y, torch.cos(a), torch.sin(a)


STATIC_STEP = 5  # the schedule step the static case runs


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "seed": seed}
    if kind in ("frames", "field", "blobs", "neighbours"):
        side = case["side"]
        s["params"] = _params(case, seed)
        s["field"] = Field2D(side, side, D, True, case["agents"])
    if kind == "blobs":
        x, y, hx, hy = workloads.clustered(case["agents"], case["side"], blobs=case["blobs"],
                                           seed=seed)
        s["agents"] = (np.arange(case["agents"], dtype=np.uint32), x, y, hx, hy)
    elif kind == "neighbours":
        s["field"].init_uniform(case["agents"], seed, 1)
        s["field"].lazy_update()
        s["field"].sync()
        # the caller's arrays, with room for half as many ids again as a
        # uniform field has
        near = 1.0 + _density(case) * math.pi * RADIUS * RADIUS
        s["row_ptr"] = np.zeros(case["agents"] + 1, np.uint32)
        s["ids"] = np.zeros(int(1.5 * near * case["agents"]) + 1024, np.uint32)
        s["total"] = ctypes.c_size_t()
    elif kind in ("ensemble", "serve"):
        s["specs"] = _specs(case, seed)
        n, steps = _sizes(case)
        s["base"] = np.concatenate([[0], np.cumsum(n)])
        s["out"] = _result(sum(n))
        s["requests"] = [workloads.Request(0.0, sp, st) for sp, st in zip(s["specs"], steps)]
    elif kind == "static":
        n, side = case["agents"], case["side"]
        s["desc"] = _abi.FieldDesc(side, side, D, 1, n, 0, 0, 0)
        s["params"] = _params(case, seed)
        s["in"] = _static_inputs(case, seed)
        s["out_ids"] = torch.empty(n, dtype=torch.int32, device="cuda")
        s["out"] = torch.empty((4, n), dtype=torch.float32, device="cuda")
        s["by_id"] = torch.empty((4, n), dtype=torch.float32, device="cuda")
    return s


def _collect(s, i, birds):
    """Run i's birds by id (an ensemble's read gives them in any order)."""
    lo, hi = s["base"][i], s["base"][i + 1]
    for k in STATE[1:]:
        s["out"][k][lo:hi][birds["id"]] = birds[k]


def _signed(birds):
    """Ids as int32, which every array library can index with."""
    return dict(birds, id=birds["id"].view(np.int32))


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "field":
        f = s["field"]
        f.init_uniform(case["agents"], s["seed"], 1)
        f.schedule_run(s["params"], 0, case["steps"])
        return _signed(f.read_agents())
    if kind == "frames":
        f = s["field"]
        f.init_uniform(case["agents"], s["seed"], 1)
        for k in range(case["steps"]):
            f.schedule_run(s["params"], k, 1)
            birds = f.read_agents()
        return _signed(birds)
    if kind == "blobs":
        f = s["field"]
        f.set_object_locations(*s["agents"])
        f.schedule_run(s["params"], 0, case["steps"])
        return _signed(f.read_agents())
    if kind == "neighbours":
        _abi.check(lib().kg_neighbor_sets(
            s["field"]._h, RADIUS, _abi.u32p(s["row_ptr"]), _abi.u32p(s["ids"]), len(s["ids"]),
            ctypes.byref(s["total"])))
        return [v.view(np.int32) for v in (s["row_ptr"], s["ids"])] + [s["total"].value]
    if kind == "ensemble":
        with Ensemble() as ens:
            ids = ens.admit(s["specs"])
            ens.run(case["steps"])
            for i, rid in enumerate(ids):
                _collect(s, i, ens.read(rid))
        return s["out"]
    if kind == "serve":
        done = serve.Server(32 << 30, keep_state=True).serve(s["requests"])
        for c in done:
            _collect(s, c.index, c.state)
        return s["out"]
    # static: one step, then the birds by id as the caller keeps them
    n = case["agents"]
    _abi.check(lib().kg_schedule_step_static(
        ctypes.byref(s["desc"]), ctypes.byref(s["params"].c()), STATIC_STEP,
        *[_ptr(t) for t in s["in"]], n, _ptr(s["out_ids"]), *[_ptr(t) for t in s["out"]], None))
    s["by_id"][:, s["out_ids"].long()] = s["out"]
    return s["by_id"]


def _step_work(agents, steps, density):
    """State (20 B) read once and written once per agent and step; about 20
    operations per neighbour and 100 per agent."""
    near = max(1.0, density * math.pi * RADIUS * RADIUS)
    return {"bytes": 40.0 * agents * steps, "flops": agents * steps * (100.0 + 20.0 * near)}


def work(case):
    kind = case["kind"]
    if kind in ("ensemble", "serve"):
        n, steps = _sizes(case)
        if kind == "ensemble":
            steps = [case["steps"]] * len(n)
        return _step_work(sum(a * b for a, b in zip(n, steps)), 1, DENSE)
    n, density = case["agents"], _density(case)
    if kind == "neighbours":
        near = 1.0 + density * math.pi * RADIUS * RADIUS
        return {"bytes": n * (12.0 + 8.0 + 4.0 * near), "flops": n * 10.0 * near}
    if kind == "blobs":
        density = 0.8 * n / case["blobs"] / (4.0 * math.pi * 200.0 ** 2)
    return _step_work(n, case.get("steps", 1), density)


# ---- one step in 64 bits --------------------------------------------------

PHILOX_M = (0xD2511F53, 0xCD9E8D57)
PHILOX_W = (0x9E3779B9, 0xBB67AE85)
TAG_STEP = 0x53544550


def _philox_uniforms(ids, step, seed):
    """The two uniforms of each bird: Philox4x32-10 of {id, step, STEP}."""
    c = [ids.astype(np.uint64), np.full(len(ids), step & 0xFFFFFFFF, np.uint64),
         np.full(len(ids), step >> 32, np.uint64), np.full(len(ids), TAG_STEP, np.uint64)]
    k = [seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF]
    low = np.uint64(0xFFFFFFFF)
    for r in range(10):
        p0, p1 = c[0] * np.uint64(PHILOX_M[0]), c[2] * np.uint64(PHILOX_M[1])
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k[0]), p1 & low,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k[1]), p0 & low]
        k = [(k[0] + PHILOX_W[0]) & 0xFFFFFFFF, (k[1] + PHILOX_W[1]) & 0xFFFFFFFF]
    return [(v >> np.uint64(8)).astype(np.float64) * 2.0 ** -24 for v in c[:2]]


def exact(case, seed):
    """The static step's birds by id in float64; cells and the torus are
    those of the f32 positions.  A run of many steps has no such value: a
    rounding travels from bird to bird."""
    if case["kind"] != "static":
        return None
    n = case["agents"]
    ids, x32, y32, hx, hy = [t.cpu().numpy() for t in _static_inputs(case, seed)]
    side = float(np.float32(case["side"]))
    d32 = np.float32(D)
    d = float(d32)
    cells = int(np.ceil(np.float32(side) / d32))
    order = np.lexsort((ids, np.floor(y32 / d32), np.floor(x32 / d32)))
    ids, x32, y32, hx, hy = [v[order] for v in (ids, x32, y32, hx, hy)]
    cx = np.floor(x32 / d32).astype(np.int64)
    cy = np.floor(y32 / d32).astype(np.int64)
    x, y, hx, hy = [v.astype(np.float64) for v in (x32, y32, hx, hy)]
    start = np.searchsorted(cx * (cells + 1) + cy, np.arange((cells + 1) ** 2 + 1))
    reach = int(math.floor(RADIUS / d))

    def axis(a, b):
        v = a - b
        return np.where(v > side / 2, v - side, np.where(v < -side / 2, v + side, v))

    acc = np.zeros((6, n))
    count = np.zeros(n)
    for i in range(-reach, reach + 1):
        for j in range(-reach, reach + 1):
            bx, by = cx + i, cy + j
            at = np.nonzero((bx >= 0) & (bx < cells) & (by >= 0) & (by < cells))[0]
            bx, by = bx[at], by[at]
            px, py = x[at], y[at]
            # check_circle: the cell's corners against the radius
            ex = [axis(bx * d, px) ** 2, axis(np.minimum(bx * d + d, side), px) ** 2]
            ey = [axis(by * d, py) ** 2, axis(np.minimum(by * d + d, side), py) ** 2]
            inside = np.maximum(*ex) + np.maximum(*ey) <= RADIUS ** 2
            beyond = np.minimum(*ex) + np.minimum(*ey) > RADIUS ** 2
            lo, hi = start[bx * (cells + 1) + by], start[bx * (cells + 1) + by + 1]
            hi = np.where(beyond, lo, hi)
            for k in range(int((hi - lo).max(initial=0))):
                m = np.nonzero(lo + k < hi)[0]
                e, b = lo[m] + k, at[m]
                dx, dy = axis(x[b], x[e]), axis(y[b], y[e])
                s = dx * dx + dy * dy
                ok = (inside[m] | (s <= RADIUS ** 2)) & (e != b)
                e, b, dx, dy, s = e[ok], b[ok], dx[ok], dy[ok], s[ok]
                for q, v in enumerate((dx / (s * s + 1.0), dy / (s * s + 1.0), dx, dy, hx[e],
                                       hy[e])):
                    acc[q][b] += v
                count[b] += 1
    c = np.maximum(count, 1.0)
    acc /= c
    r1, r2 = _philox_uniforms(ids, STATIC_STEP, seed)
    rx, ry = r1 * 2.0 - 1.0, r2 * 2.0 - 1.0
    rn = np.sqrt(rx * rx + ry * ry)
    p = _params(case, seed)
    vx = (p.cohesion * -acc[2] / 10.0 + p.avoidance * 400.0 * acc[0]
          + p.consistency * acc[4] / c + p.randomness * 0.05 * rx / rn + p.momentum * hx)
    vy = (p.cohesion * -acc[3] / 10.0 + p.avoidance * 400.0 * acc[1]
          + p.consistency * acc[5] / c + p.randomness * 0.05 * ry / rn + p.momentum * hy)
    norm = np.sqrt(vx * vx + vy * vy)
    norm = np.where(norm > 0, norm, 1.0)
    vx, vy = vx / norm * p.jump, vy / norm * p.jump
    out = np.empty((4, n))
    out[:, ids] = np.stack([np.mod(x + vx, side), np.mod(y + vy, side), vx, vy])
    return torch.from_numpy(out)
