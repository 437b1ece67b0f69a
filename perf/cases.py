"""The workloads this framework's speed is measured on.

Each case is work a user's program has the framework do, through its Python
entry points (openabl_amd.Simulation, Ensemble and generated step programs):

  kind "run"       the body of a model's main(): upload the agents, simulate a
                   number of timesteps, download the agents (what a program
                   does for each run of a sweep);
  kind "ensemble"  many uneven runs of one program kept on the device, advanced
                   together by a number of timesteps and read back.

Models, sizes and launch settings are those of the examples, tests and
benchmark of this repository.  `exact` restates each model in plain torch in
64 bits.  A distance is the language's: the square root rounded to single
precision (the runtime's sqrtf) in every float type.
"""
import math

import numpy as np
import torch

from openabl_amd import AGENTS, Simulation, codegen, record_dtype
from openabl_amd.ensemble import Ensemble

# cells of half the near radius and tight LDS tiles: the launch settings of the
# benchmark's boids2d workload; everything else runs at the defaults
BOIDS_TUNED = {"hip.cell_scale": 2, "hip.tile": 1, "hip.block": 256, "hip.lds_slack": 1.25,
               "hip.nlist": 1, "hip.skin": 0.05}
# the benchmark's settings for clustered circle3d: one thread per agent
CIRCLE3D_UNTILED = {"hip.cell_scale": 2, "hip.tile": 0, "hip.block": 256}
CONFIGS = {"default": {}, "boids_tuned": BOIDS_TUNED, "circle3d_untiled": CIRCLE3D_UNTILED}

# generated programs carry their parameters as constants: the environment is
# that of this many agents whatever number is uploaded
GENERATED_AGENTS = {"bench_boids2d_cfg": 1048576}
BOIDS_DENSITY = 0.065536


def fold6(x):
    """A derived constant as the compiler folds it (six significant digits)."""
    return float("%.6g" % x)


def listed():
    return [
        # the smallest model at its defaults: launches and latency
        {"name": "circle_1k", "kind": "run", "model": "circle", "precision": "f64", "agents": 1000,
         "steps": 20, "rho": 0.05, "r": 5.0, "config": "default"},
        # the model with births, deaths and a sequential step, at its defaults:
        # thirteen step functions and several read-backs per timestep
        {"name": "predator_prey_3k", "kind": "run", "model": "predator_prey", "precision": "f64",
         "agents": 3200, "steps": 20, "prey": 0.35, "predators": 0.025, "config": "default"},
        # a middling flock (the model's own size) that moves ten times as far per
        # timestep: re-sorted now and then, and denser where flocks form, as the
        # model gets in any long run
        {"name": "boids2d_64k", "kind": "run", "model": "boids2d", "precision": "f64",
         "agents": 65536, "steps": 300, "time_scale": 0.005, "config": "default"},
        # the benchmark's workload: a million boids, 200 timesteps
        {"name": "boids2d_1m", "kind": "run", "model": "boids2d", "precision": "f64",
         "agents": 1048576, "steps": 200, "time_scale": 0.0005, "config": "boids_tuned"},
        # single precision (use_float), a ragged number of agents
        {"name": "boids2d_f32_300k", "kind": "run", "model": "boids2d", "precision": "f32",
         "agents": 300007, "steps": 100, "time_scale": 0.0005, "config": "default"},
        # agents that change cells on every timestep: a re-sort per timestep
        {"name": "circle_1m", "kind": "run", "model": "circle", "precision": "f64",
         "agents": 1000003, "steps": 40, "rho": 0.1024, "r": 2.5, "config": "default"},
        # uneven density in 3-D, compensated single precision, tuned settings
        {"name": "clustered_f32c_1m", "kind": "run", "model": "circle3d", "precision": "f32c",
         "agents": 1048576, "steps": 5, "clusters": 64, "config": "circle3d_untiled"},
        # uneven density in 3-D as a program at the defaults runs it
        {"name": "clustered_f64_200k", "kind": "run", "model": "circle3d", "precision": "f64",
         "agents": 200003, "steps": 10, "clusters": 16, "config": "default"},
        # a cellular automaton: agents that never move, one byte of state
        {"name": "life_1m", "kind": "run", "model": "game_of_life", "precision": "f64",
         "agents": 1048576, "steps": 100, "alive": 0.3, "config": "default"},
        # births and deaths with a larger population
        {"name": "predator_prey_250k", "kind": "run", "model": "predator_prey", "precision": "f64",
         "agents": 250000, "steps": 10, "prey": 0.4, "predators": 0.04, "config": "default"},
        # a parameter study: uneven flocks in one launch, replayed as a graph (the
        # members live on from pass to pass: a small time step keeps them alike)
        {"name": "ensemble_30", "kind": "ensemble", "model": "boids2d", "precision": "f64",
         "members": 30, "least": 1000, "most": 65536, "steps": 100, "time_scale": 0.0001,
         "config": "default"},
        # the compiler's output for the benchmark's model, at the defaults
        {"name": "generated_boids2d_1m", "kind": "run", "model": "boids2d",
         "program": "bench_boids2d_cfg", "precision": "f64", "agents": 1048576, "steps": 50,
         "time_scale": 0.0005, "config": "default"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["circle", "circle", "boids2d", "boids2d", "clustered", "uniform3d", "life",
                       "predator_prey", "predator_prey", "ensemble", "generated"])
    if what == "circle":
        # the model amplifies a rounding tenfold in a few timesteps: short runs
        # in single precision
        rho, r = rng.choice([(0.05, 5.0), (0.1024, 2.5)])
        precision = rng.choice(["f64", "f64", "f32", "f32c"])
        return {"kind": "run", "model": "circle", "precision": precision,
                "agents": _log_int(rng, 500, 1000003),
                "steps": rng.randint(5, 40 if precision == "f64" else 10), "rho": rho, "r": r,
                "config": "default"}
    if what == "boids2d":
        precision = rng.choice(["f64", "f64", "f32", "f32c"])
        return {"kind": "run", "model": "boids2d", "precision": precision,
                "agents": _log_int(rng, 1000, 1048576),
                "steps": rng.randint(20, 200 if precision == "f64" else 100),
                "time_scale": rng.choice([0.0005, 0.005]) if precision == "f64" else 0.0005,
                "config": rng.choice(["default", "default", "boids_tuned"])}
    if what == "clustered":
        n = _log_int(rng, 5000, 1048576)
        return {"kind": "run", "model": "circle3d", "precision": rng.choice(["f64", "f32c", "f32"]),
                "agents": n, "steps": rng.randint(2, 5), "clusters": max(1, n // 14000),
                "config": "circle3d_untiled" if n > 250000 else rng.choice(["default", "circle3d_untiled"])}
    if what == "uniform3d":
        return {"kind": "run", "model": "circle3d", "precision": rng.choice(["f64", "f32", "f32c"]),
                "agents": _log_int(rng, 1000, 200003), "steps": rng.randint(2, 5), "clusters": 0,
                "config": "default"}
    if what == "life":
        return {"kind": "run", "model": "game_of_life", "precision": rng.choice(["f64", "f32"]),
                "agents": _log_int(rng, 400, 1048576), "steps": rng.randint(20, 100),
                "alive": rng.choice([0.1, 0.3]), "config": "default"}
    if what == "predator_prey":
        prey, pred = rng.choice([(0.35, 0.025), (0.4, 0.04)])
        return {"kind": "run", "model": "predator_prey", "precision": "f64",
                "agents": _log_int(rng, 1000, 250000), "steps": rng.randint(5, 20), "prey": prey,
                "predators": pred, "config": "default"}
    if what == "ensemble":
        return {"kind": "ensemble", "model": "boids2d", "precision": rng.choice(["f64", "f32"]),
                "members": rng.randint(4, 30), "least": 1000, "most": rng.choice([8192, 65536]),
                "steps": rng.randint(20, 100), "time_scale": 0.0001, "config": "default"}
    return {"kind": "run", "model": "boids2d", "program": "bench_boids2d_cfg",
            "precision": rng.choice(["f64", "f32"]), "agents": _log_int(rng, 100000, 1048576),
            "steps": rng.randint(10, 50), "time_scale": 0.0005, "config": "default"}


# ---- parameters -------------------------------------------------------------------


def box_of(case):
    """Side of the environment."""
    n = GENERATED_AGENTS.get(case.get("program"), case.get("agents", 0))
    if case["model"] == "circle":
        return fold6(math.sqrt(n / case["rho"]))
    if case["model"] == "circle3d":
        return fold6(float(np.cbrt(n / circle3d_rho(case))))
    if case["model"] == "boids2d":
        return fold6(math.sqrt(n / BOIDS_DENSITY))
    if case["model"] == "predator_prey":
        return fold6(math.sqrt(n / 1600.0))
    return float(math.isqrt(n))


def circle3d_rho(case):
    return 1048576 / 1e9 if case["clusters"] else 0.05


def circle3d_r(case):
    return 4.0 if case["clusters"] else 5.0


def params_of(case):
    n = case["agents"]
    if case["model"] == "circle":
        return {"num_agents": n, "rho": case["rho"], "r": case["r"]}
    if case["model"] == "circle3d":
        return {"num_agents": n, "rho": circle3d_rho(case), "r": circle3d_r(case),
                "num_clusters": case["clusters"]}
    if case["model"] == "boids2d":
        return {"num_agents": n, "agent_density": BOIDS_DENSITY, "time_scale": case["time_scale"]}
    if case["model"] == "predator_prey":
        return {"num_agents": n, "prey_fraction": case["prey"], "predator_fraction": case["predators"]}
    return {"num_agents": n, "alive_fraction": case["alive"]}


def ensemble_sizes(case):
    u = np.random.default_rng(case["members"]).uniform(0.0, 1.0, case["members"])
    return (case["least"] * (case["most"] / case["least"]) ** u).astype(int).tolist()


def ensemble_members(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n in ensemble_sizes(case):
        w = rng.uniform(0.5, 2.0, 3)
        out.append({"num_agents": n, "agent_density": 0.065, "max_pos": fold6(math.sqrt(n / 0.065)),
                    "time_scale": case["time_scale"], "steer_scale": float(w[0]),
                    "collision_scale": float(w[1]), "match_scale": float(w[2])})
    return out


# ---- inputs -----------------------------------------------------------------------


def inputs_of(case, seed):
    """One record array per agent type: what main() creates before simulate()."""
    rng = np.random.default_rng(seed)
    model, n, box = case["model"], case["agents"], box_of(case)
    dts = [record_dtype(members, case["precision"]) for _, members in AGENTS[model]]
    if model == "predator_prey":
        npred, nprey = int(case["predators"] * n), int(case["prey"] * n)
        pred, prey, grass = (np.zeros(k, dt) for k, dt in zip((npred, nprey, n - npred - nprey), dts))
        for rec, gain in ((pred, 35), (prey, 60)):
            rec["pos"] = rng.uniform(0.0, box, rec["pos"].shape)
            phi = rng.uniform(0.0, 2.0 * math.pi, len(rec))
            rec["dir"] = np.stack([np.sin(phi), np.cos(phi)], 1)
            rec["life"] = gain + rng.integers(0, 11, len(rec))
        grass["pos"] = rng.uniform(0.0, box, grass["pos"].shape)
        grass["avail"] = 1
        return [pred, prey, grass]
    if model == "game_of_life":
        side = math.isqrt(n)
        rec = np.zeros(side * side, dts[0])
        x, y = np.divmod(np.arange(side * side), side)
        rec["pos"] = np.stack([x + 0.5, y + 0.5], 1)
        rec["alive"] = rng.random(side * side) < case["alive"]
        return [rec]
    rec = np.zeros(n, dts[0])
    if model == "circle3d" and case["clusters"]:
        each = int(0.8 * n) // case["clusters"]
        pos = rng.uniform(0.0, box, (n, 3))
        centres = np.repeat(rng.uniform(0.0, box, (case["clusters"], 3)), each, 0)
        pos[: len(centres)] = np.clip(centres + rng.normal(0.0, 20.0, centres.shape), 0.0, box)
        rec["pos"] = pos
    else:
        rec["pos"] = rng.uniform(0.0, box, rec["pos"].shape)
    if model == "boids2d":
        rec["velocity"] = rng.uniform(-1.0, 1.0, rec["velocity"].shape)
    return [rec]


def prepare(case, seed):
    config = CONFIGS[case["config"]]
    if case["kind"] == "ensemble":
        ens = Ensemble(case["model"], case["precision"], ensemble_members(case, seed), config=config)
        ens.init(0xDEADBEEF ^ seed, 0xBEEFDEAD)
        return {"case": case, "ens": ens}
    if "program" in case:
        codegen.load_program(codegen.program_dir(case["program"]))
        sim = Simulation(case["program"], case["precision"], config=config)
    else:
        sim = Simulation(case["model"], case["precision"], params=params_of(case), config=config)
    recs = inputs_of(case, seed)
    return {"case": case, "sim": sim, "recs": recs, "dts": [r.dtype for r in recs]}


# the state a program reads back, per model and agent type
READ = {"circle": [["pos"]], "circle3d": [["pos"]], "boids2d": [["pos", "velocity"]],
        "game_of_life": [["alive"]],
        "predator_prey": [["pos", "dir", "steer", "life"], ["pos", "dir", "steer", "life"],
                          ["dead_cycles", "avail"]]}


def outputs_of(case, recs):
    out = [{name: rec[name] for name in names} for names, rec in zip(READ[case["model"]], recs)]
    if case["model"] == "predator_prey":
        # a table of fixed length per mover type, whatever number is alive
        for cols in out[:2]:
            for name, col in cols.items():
                table = np.zeros((case["agents"] // 2,) + col.shape[1:], col.dtype)
                table[: len(col)] = col
                cols[name] = table
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "ensemble":
        ens = state["ens"]
        ens.simulate(case["steps"])
        return [outputs_of(case, [ens.download(m)])[0] for m in range(ens.members)]
    sim = state["sim"]
    for t, rec in enumerate(state["recs"]):
        sim.upload(rec, t)
    sim.simulate(case["steps"])
    return outputs_of(case, [sim.download(dt, t) for t, dt in enumerate(state["dts"])])


# ---- what the work cannot do without ------------------------------------------------


def work(case):
    """A timestep reads every member of every agent once and writes each member
    its step functions assign once; a run also takes the records in and gives
    them back.  Operations are those of the accepted neighbours (expected
    number, agents uniform or in their clusters) and of each agent's update."""
    fb = 4 if case["precision"] == "f32" else 8
    steps, model = case["steps"], case["model"]
    if case["kind"] == "ensemble":
        n = sum(ensemble_sizes(case))
    else:
        n = case["agents"]
    moved = 2 if case["kind"] == "run" else 1
    if model == "boids2d":
        rec = 2 * 2 * fb
        if case["precision"] == "f32c":
            rec = 2 * 8 + 2 * 4
        density = n / box_of(case) ** 2 if case["kind"] != "ensemble" else 0.065
        near, per_pair, per_agent = math.pi * 100.0 * density, 11, 50
        step_bytes = 2 * rec
    elif model == "circle":
        rec = 2 * fb
        near, per_pair, per_agent = math.pi * (2 * case["r"]) ** 2 * case["rho"], 14, 4
        step_bytes = 2 * rec
    elif model == "circle3d":
        rec = 3 * fb
        ball = 4.0 / 3.0 * math.pi * (2 * circle3d_r(case)) ** 3
        near = ball * circle3d_rho(case)
        if case["clusters"]:
            # mean density of a Gaussian cluster, sigma 20, seen by its agents
            near = 0.2 * near + 0.8 * ball * 0.8 * n / case["clusters"] / (4.0 * math.pi * 400.0) ** 1.5
        per_pair, per_agent = 18, 6
        step_bytes = 2 * rec
    elif model == "game_of_life":
        rec, near, per_pair, per_agent = 1, 9.0, 1, 2
        step_bytes = 2 * rec
    else:
        movers, grass = case["prey"] + case["predators"], 1.0 - case["prey"] - case["predators"]
        rec = movers * (6 * fb + 4) + grass * (2 * fb + 5)
        # prey in an agent's cohesion disk, and the smaller disks
        near, per_pair, per_agent = movers * math.pi * 0.12 ** 2 * 1600.0 * movers, 14, 60
        step_bytes = rec + movers * (6 * fb + 4) + grass * 5
    flops = steps * n * (near * per_pair + per_agent)
    return {"bytes": float(n * (steps * step_bytes + moved * rec)), "flops": float(flops)}


def tolerance(case):
    """About four times what a run differs by from the same run visiting its
    neighbours in index order, or from `exact`: roundings, amplified by the
    model, and now and then a pair on the other side of a radius."""
    if case["model"] == "game_of_life":
        return "exact"
    single = {"boids2d": {"f32": 0.02, "f32c": 0.02}, "circle": {"f32": 2e-3, "f32c": 1e-5},
              "circle3d": {"f32": 5e-3, "f32c": 2e-5}}
    if case["precision"] != "f64":
        return {"rel": single[case["model"]][case["precision"]], "max": 0.99}
    return {"boids2d": {"rel": 1e-6, "max": 1e-3}, "circle": {"rel": 1e-9, "max": 1e-6},
            "circle3d": {"rel": 1.2e-7, "max": 1e-4},
            "predator_prey": {"rel": 1e-9, "max": 1e-6, "differ": 1e-4}}[case["model"]]


# ---- the models in 64 bits ----------------------------------------------------------


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _dist(s):
    """dist() of the language from a square sum."""
    return torch.sqrt(s.to(torch.float32)).to(torch.float64)


class _Grid:
    """Points binned into cells of side r (one grid per group)."""

    def __init__(self, pos, r, box, group=None, groups=1):
        self.pos, self.r, self.group = pos, r, group
        self.n = max(1, int(box / r))
        self.side = box / self.n
        self.dim = pos.shape[1]
        key = self._key(self.cells(pos), group)
        self.order = torch.argsort(key, stable=True)
        count = torch.bincount(key, minlength=groups * self.n ** self.dim)
        self.start = torch.cat([count.new_zeros(1), count.cumsum(0)])

    def cells(self, pos):
        return (pos / self.side).floor().long().clamp(0, self.n - 1)

    def _key(self, cell, group):
        key = torch.zeros_like(cell[:, 0]) if group is None else group
        for d in range(self.dim):
            key = key * self.n + cell[:, d]
        return key

    def pairs(self, pos, group=None):
        """(i, j, s): every point j within r of query point i, its square
        distance s; in pieces, one per row of cells beside the query's cell."""
        cell = self.cells(pos)
        for off in np.ndindex(*([3] * (self.dim - 1))):
            c = cell.clone()
            ok = torch.ones(len(pos), dtype=torch.bool, device=pos.device)
            for d, o in enumerate(off):
                c[:, d] += o - 1
                ok &= (c[:, d] >= 0) & (c[:, d] < self.n)
            q = ok.nonzero()[:, 0]
            c = c[q]
            last = c[:, self.dim - 1].clone()
            g = None if group is None else group[q]
            c[:, self.dim - 1] = (last - 1).clamp(min=0)
            a = self.start[self._key(c, g)]
            c[:, self.dim - 1] = (last + 1).clamp(max=self.n - 1)
            b = self.start[self._key(c, g) + 1]
            total = torch.cumsum(b - a, 0)
            # at most about 2**27 candidates at a time
            at = 0
            while at < len(q):
                base = int(total[at - 1]) if at else 0
                end = max(at + 1, int(torch.searchsorted(total, base + (1 << 27))))
                num = (b - a)[at:end]
                i = torch.repeat_interleave(q[at:end], num)
                first = torch.repeat_interleave(a[at:end] - (total[at:end] - num - base), num)
                j = self.order[first + torch.arange(len(i), device=pos.device)]
                e = self.pos[j] - pos[i]
                s = (e * e).sum(1)
                near = _dist(s) <= self.r
                yield i[near], j[near], s[near]
                at = end


def _circle_step(pos, box, r, k_rep=0.05, k_att=0.01):
    new = pos.clone()
    for i, j, s in _Grid(pos, 2.0 * r, box).pairs(pos):
        d = _dist(s)
        k = d != 0
        i, j, d = i[k], j[k], d[k][:, None]
        e = pos[j] - pos[i]
        new.index_add_(0, i, torch.where(d > r, e * (k_att * (2.0 * r - d)) / d, -e * k_rep))
    return new.clamp(1.0, box - 1.0)


def _boids_step(pos, vel, top, group, groups, weights, time_scale):
    """top: side of each agent's box; weights: steer, collision, match of each agent."""
    n = len(pos)
    near, close = (torch.zeros((n, k), dtype=pos.dtype, device=pos.device) for k in (5, 3))
    for i, j, s in _Grid(pos, 10.0, float(top.max()), group, groups).pairs(pos, group):
        one = torch.ones_like(s)[:, None]
        near.index_add_(0, i, torch.cat([pos[j], vel[j], one], 1))
        k = _dist(s) < 2.0
        close.index_add_(0, i[k], torch.cat([pos[j[k]], one[k]], 1))
    some = near[:, 4:] > 0
    change = torch.where(some, (near[:, :2] / near[:, 4:] - pos) * weights[:, 0:1], torch.zeros_like(pos))
    change += torch.where(some, near[:, 2:4] / near[:, 4:] * weights[:, 2:3], torch.zeros_like(pos))
    change += torch.where(close[:, 2:] > 0, (pos - close[:, :2] / close[:, 2:].clamp(min=1.0)) * weights[:, 1:2],
                          torch.zeros_like(pos))
    vel = vel + change * 0.15
    speed = _dist((vel * vel).sum(1))[:, None]
    vel = torch.where(speed > 2.0, vel / speed * 2.0, vel)
    pos = pos + vel * time_scale
    top = top[:, None]
    pos = torch.where(pos < 0.0, top.expand_as(pos), torch.where(pos > top, torch.zeros_like(pos), pos))
    return pos, vel


def _life_step(alive):
    p = np.pad(alive, 1)
    h, w = alive.shape
    living = sum(p[y:y + h, x:x + w] for y in range(3) for x in range(3)) - alive
    return ((living == 3) | ((alive == 1) & (living == 2))).astype(np.int64)


def _mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _step_random(t, step, ids):
    """random(1.0), first call of step function `step` at timestep t by each agent."""
    with np.errstate(over="ignore"):
        z = _mix64(np.array([0x5EED], np.uint64) + np.uint64(0x9E3779B97F4A7C15) * np.uint64(t + 1))
        z = _mix64(_mix64(z ^ np.uint64(step << 32)) + ids.cpu().numpy().astype(np.uint64))
    return torch.from_numpy(z.astype(np.float64) / 18446744073709551615.0).to(ids.device)


class _Movers:
    """Predators or prey: columns and ids."""

    def __init__(self, rec, dev):
        self.c = {k: torch.from_numpy(np.ascontiguousarray(rec[k])).to(dev) for k in ("pos", "dir", "steer", "life")}
        self.id = torch.arange(len(rec), device=dev)
        self.next = len(rec)

    def keep(self, mask):
        self.c = {k: v[mask] for k, v in self.c.items()}
        self.id = self.id[mask]

    def move(self, scale, env):
        v = self.c["dir"] + self.c["steer"]
        speed = _dist((v * v).sum(1))[:, None]
        v = torch.where(speed > 1.0, v / speed, v)
        self.c["pos"] = (self.c["pos"] + scale(v)).clamp(0.0, env)
        self.c["dir"] = v
        self.c["life"] = self.c["life"] - 1

    def breed(self, draws, p):
        born = draws < p
        life = torch.where(born, self.c["life"] // 2, self.c["life"])
        child = {"pos": self.c["pos"][born], "dir": self.c["dir"][born] * -1.0,
                 "steer": self.c["steer"][born] * -1.0, "life": life[born]}
        self.c["life"] = life
        self.c = {k: torch.cat([v, child[k]]) for k, v in self.c.items()}
        k = int(born.sum())
        self.id = torch.cat([self.id, self.next + torch.arange(k, device=self.id.device)])
        self.next += k


def _avoid(pos, grid, other, radius, apart):
    """Sum of (pos - other) * (radius / distance) over the others closer than radius."""
    out = torch.zeros_like(pos)
    for i, j, s in grid.pairs(pos):
        d = _dist(s)
        k = (d < radius) & (d > 0.0)
        if apart:
            k &= (other[j] != pos[i]).any(1)
        i, j, d = i[k], j[k], d[k]
        out.index_add_(0, i, (pos[i] - other[j]) * (radius / d)[:, None])
    return out


def _predator_prey(recs, steps, env, dev):
    pred, prey = _Movers(recs[0], dev), _Movers(recs[1], dev)
    gpos = torch.from_numpy(np.ascontiguousarray(recs[2]["pos"])).to(dev)
    dead = torch.zeros(len(gpos), dtype=torch.int64, device=dev)
    avail = torch.ones(len(gpos), dtype=torch.bool, device=dev)
    grass = _Grid(gpos, 0.02, env)
    for t in range(steps):
        # the nearest prey a predator sees
        p, q = pred.c["pos"], prey.c["pos"]
        best = torch.full((len(p),), 0.1, dtype=torch.float64, device=dev)
        seen = torch.full((len(p),), -1, dtype=torch.int64, device=dev)
        for i, j, s in _Grid(q, 0.1, env).pairs(p):
            d = _dist(s)
            least = best.clone().scatter_reduce_(0, i, d, "amin")
            k = (d == least[i]) & (d < best[i])
            seen[i[k]] = j[k]
            best = least
        steer = torch.where((seen >= 0)[:, None], q[seen.clamp(min=0)] - p, torch.zeros_like(p))
        away = _avoid(q, _Grid(p, 0.1, env), p, 0.1, False)
        flock = _Grid(q, 0.12, env)
        total = torch.zeros((len(q), 3), dtype=torch.float64, device=dev)
        for i, j, s in flock.pairs(q):
            total.index_add_(0, i, torch.cat([q[j], torch.ones_like(s)[:, None]], 1))
        prey.c["steer"] = away + (total[:, :2] / total[:, 2:] - q) + _avoid(q, flock, q, 0.035, True)
        pred.c["steer"] = steer + _avoid(p, _Grid(p, 0.035, env), p, 0.035, True)
        prey.move(lambda v: v * 0.0015 * 1.0, env)
        pred.move(lambda v: v * 0.0015 * 2.0 * 1.0, env)
        # eat or starve
        for i, j, _ in grass.pairs(prey.c["pos"]):
            prey.c["life"].index_add_(0, i, 60 * avail[j].to(prey.c["life"].dtype))
        prey.keep(prey.c["life"] >= 1)
        q = _Grid(prey.c["pos"], 0.02, env)
        for i, j, _ in q.pairs(pred.c["pos"]):
            pred.c["life"].index_add_(0, i, torch.full_like(j, 35, dtype=pred.c["life"].dtype))
        pred.keep(pred.c["life"] >= 1)
        eaten = torch.zeros_like(avail)
        for i, j, s in q.pairs(gpos):
            eaten[i[_dist(s) < 0.02]] = True
        eaten &= avail
        dead[eaten] = 0
        avail &= ~eaten
        gone = torch.zeros(len(prey.id), dtype=torch.bool, device=dev)
        for i, j, s in _Grid(pred.c["pos"], 0.02, env).pairs(prey.c["pos"]):
            gone[i[_dist(s) < 0.02]] = True
        prey.keep(~gone)
        pred.breed(_step_random(t, 10, pred.id), 0.001)
        prey.breed(_step_random(t, 11, prey.id), 0.005)
        grown = dead == 60
        old = avail.clone()
        dead = torch.where(old, torch.where(grown, torch.zeros_like(dead), dead), dead + 1)
        avail |= grown
    movers = [{k: v.cpu().numpy() for k, v in m.c.items()} for m in (pred, prey)]
    return movers + [{"dead_cycles": dead.to(torch.int32).cpu().numpy(), "avail": avail.to(torch.uint8).cpu().numpy()}]


def exact(case, seed):
    model, steps, dev = case["model"], case["steps"], _device()
    if model == "game_of_life":
        rec = inputs_of(case, seed)[0]
        side = math.isqrt(case["agents"])
        alive = rec["alive"].reshape(side, side).astype(np.int64)
        for _ in range(steps):
            alive = _life_step(alive)
        return [{"alive": alive.reshape(-1).astype(np.uint8)}]
    if model == "predator_prey":
        return outputs_of(case, _predator_prey(inputs_of(case, seed), steps, box_of(case), dev))

    def up(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev, torch.float64)

    if case["kind"] == "ensemble":
        params = ensemble_members(case, seed)
        ens = prepare(case, seed)["ens"]
        recs = [ens.download(m) for m in range(ens.members)]
    else:
        params = [{"max_pos": box_of(case), "steer_scale": 1.0, "collision_scale": 1.5, "match_scale": 1.0}]
        recs = inputs_of(case, seed)
    sizes = [len(rec) for rec in recs]
    pos = torch.cat([up(rec["pos"]) for rec in recs])
    if model != "boids2d":
        r = case["r"] if model == "circle" else circle3d_r(case)
        for _ in range(steps):
            pos = _circle_step(pos, box_of(case), r)
        return [{"pos": pos.cpu().numpy()}]
    vel = torch.cat([up(rec["velocity"]) for rec in recs])
    group = torch.repeat_interleave(torch.arange(len(sizes), device=dev), torch.tensor(sizes, device=dev))
    top = up([p["max_pos"] for p in params])[group]
    weights = up([[p["steer_scale"], p["collision_scale"], p["match_scale"]] for p in params])[group]
    for _ in range(steps):
        pos, vel = _boids_step(pos, vel, top, group, len(sizes), weights, case["time_scale"])
    return [{"pos": p.cpu().numpy(), "velocity": v.cpu().numpy()}
            for p, v in zip(torch.split(pos, sizes), torch.split(vel, sizes))]
