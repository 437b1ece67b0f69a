"""Batched ensembles: every member of a batch is bit-identical to the same
run computed alone (same parameters, generator start state, cell scale, tile
shape and list settings), with and without graph replay, with neighbour lists
(members re-sorted and rebuilt on their own schedules) and without, FP64 and
FP32."""
import math

import numpy as np
import pytest

from orclib import field_bytes, fold6

pytestmark = pytest.mark.gpu


def members(k, seed=5):
    rng = np.random.default_rng(seed)
    out = []
    for n in np.exp(rng.uniform(math.log(1000), math.log(8000), k)).astype(int):
        w = rng.uniform(0.5, 2.0, 3)
        out.append({"num_agents": int(n), "agent_density": 0.065,
                    "max_pos": fold6(math.sqrt(n / 0.065)),
                    "steer_scale": float(w[0]), "collision_scale": float(w[1]),
                    "match_scale": float(w[2])})
    return out


LISTS = {"stencil": {"hip.nlist": 0},
         # a fixed list capacity: lists that outgrow it overflow
         "lists": {"hip.nlist": 1, "hip.list_cap": 96},
         # a skin a boid at full speed crosses in three steps: rebuilds
         "lists-skin": {"hip.nlist": 1, "hip.list_cap": 96, "hip.skin": 0.0005}}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("graph,steps", [(1, 30), (1, 31), (0, 12)])
@pytest.mark.parametrize("mode", sorted(LISTS))
def test_members_equal_alone_runs(prec, graph, steps, mode):
    from openabl_amd import MEMBERS, Simulation, load_library, record_dtype
    from openabl_amd.ensemble import Ensemble, member_seed
    print(f"case ensemble members vs alone {prec} graph={graph} steps={steps} {mode}", flush=True)
    ms = members(10)
    cfg = dict({"hip.cell_scale": 2, "hip.tile": 1}, **LISTS[mode])
    ens = Ensemble("boids2d", prec, ms, config=dict(cfg, **{"hip.graph": graph}))
    ens.init(0x1234, 0x5678)
    ens.simulate(steps)
    ens.synchronize()
    dt = record_dtype(MEMBERS["boids2d"], prec)
    for m, p in enumerate(ms):
        load_library().abl_rng_seed(*member_seed(0x1234, 0x5678, m))
        sim = Simulation("boids2d", prec, params=p, config=cfg)
        sim.init_agents()
        sim.simulate(steps)
        assert field_bytes(ens.download(m)) == field_bytes(sim.download(dt)), m
        sim.close()
    ens.close()


def test_lists_follow_each_members_own_rebuilds():
    """Members whose agents move at different speeds rebuild on different
    timesteps: half the members move 50x slower (time_scale), so with a skin
    the fast ones are due every step and the slow ones every few steps; every
    member still equals its run alone, which rebuilds only when its own agents
    stray."""
    from openabl_amd import MEMBERS, Simulation, load_library, record_dtype
    from openabl_amd.ensemble import Ensemble, member_seed
    print("case ensemble lists with members on different rebuild schedules", flush=True)
    ms = members(8, seed=9)
    for k, m in enumerate(ms):
        m["time_scale"] = 0.25 if k % 2 else 0.005
    cfg = {"hip.cell_scale": 2, "hip.tile": 1, "hip.nlist": 1, "hip.list_cap": 96,
           "hip.skin": 0.02}
    ens = Ensemble("boids2d", "f64", ms, config=cfg)
    ens.init(0x1234, 0x5678)
    ens.simulate(24)
    ens.synchronize()
    dt = record_dtype(MEMBERS["boids2d"], "f64")
    for m, p in enumerate(ms):
        load_library().abl_rng_seed(*member_seed(0x1234, 0x5678, m))
        sim = Simulation("boids2d", "f64", params=p, config=cfg)
        sim.init_agents()
        sim.simulate(24)
        assert field_bytes(ens.download(m)) == field_bytes(sim.download(dt)), m
        sim.close()
    ens.close()


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("count,most", [(1, 700), (255, 3), (256, 40), (300, 40), (520, 9)])
def test_rebuild_chunks_of_many_members(count, most, graph):
    """The one-launch rebuild numbers the chunks of the members due in groups of
    members (one per thread of a block; from 257 members on two or more each):
    members of no more than one chunk, of several, of a single agent."""
    from openabl_amd import MEMBERS, Simulation, load_library, record_dtype
    from openabl_amd.ensemble import Ensemble, member_seed
    print(f"case ensemble rebuild chunks {count} {most} graph={graph}", flush=True)
    rng = np.random.default_rng(count)
    ms = [{"num_agents": int(n), "agent_density": 0.065, "max_pos": fold6(math.sqrt(n / 0.065)),
           "time_scale": 0.01} for n in rng.integers(1, most + 1, count)]
    cfg = {"hip.cell_scale": 2, "hip.tile": 1, "hip.nlist": 1, "hip.list_cap": 96, "hip.skin": 0.001}
    ens = Ensemble("boids2d", "f64", ms, config=dict(cfg, **{"hip.graph": graph}))
    ens.init(0x1234, 0x5678)
    assert ens.inspect("rebuild_launches") == 1
    ens.simulate(17)
    assert ens.inspect("rebuild_launches") == 4  # most of the first timesteps rebuilt
    ens.simulate(7)
    dt = record_dtype(MEMBERS["boids2d"], "f64")
    for m in sorted({0, count // 2, count - 1, *rng.integers(0, count, 3).tolist()}):
        load_library().abl_rng_seed(*member_seed(0x1234, 0x5678, m))
        sim = Simulation("boids2d", "f64", params=ms[m], config=cfg)
        sim.init_agents()
        sim.simulate(24)
        assert field_bytes(ens.download(m)) == field_bytes(sim.download(dt)), m
        sim.close()
    ens.close()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("graph,chunks", [(1, (90, 110, 141)), (0, (341,)), (1, (17, 1, 71, 252))])
def test_lists_grow_as_in_runs_alone(prec, graph, chunks):
    """Members whose agents draw together until their lists outgrow the capacity
    sized from their density: each enters its lists anew, with more room, on the
    timestep a run of it alone does, so capacities and bits stay the run's,
    however simulate() is called.  One member stays as it is."""
    from openabl_amd import MEMBERS, Simulation, load_library, record_dtype
    from openabl_amd.ensemble import Ensemble, member_seed
    print(f"case ensemble growing lists {prec} graph={graph} {chunks}", flush=True)
    ms = [{"num_agents": n, "agent_density": 0.065536, "max_pos": fold6(math.sqrt(n / 0.065536)),
           "time_scale": t, "steer_scale": s, "collision_scale": 1.5}
          for n, t, s in ((3001, 0.05, 3.0), (1500, 0.02, 3.0), (700, 0.0005, 1.0), (2000, 0.2, 2.0))]
    cfg = {"hip.cell_scale": 1, "hip.tile": 1, "hip.nlist": 1}
    ens = Ensemble("boids2d", prec, ms, config=dict(cfg, **{"hip.graph": graph}))
    ens.init(0x1234, 0x5678)
    first = [ens.inspect("list_capacity", m) for m in range(len(ms))]
    sims = []
    for m, p in enumerate(ms):
        load_library().abl_rng_seed(*member_seed(0x1234, 0x5678, m))
        sims.append(Simulation("boids2d", prec, params=p, config=cfg))
        sims[m].init_agents()
    dt = record_dtype(MEMBERS["boids2d"], prec)
    for n in chunks:
        ens.simulate(n)
        for m, sim in enumerate(sims):
            sim.simulate(n)
            assert field_bytes(ens.download(m)) == field_bytes(sim.download(dt)), (n, m)
    last = [ens.inspect("list_capacity", m) for m in range(len(ms))]
    assert last == [sim.inspect("list_capacity") for sim in sims]
    grown = [b > a for a, b in zip(first, last)]
    assert sum(grown) >= 2 and not grown[2], (first, last)
    for sim in sims:
        sim.close()
    ens.close()


def test_members_equal_alone_runs_while_the_rebuild_changes_form():
    """A batch whose rebuild rate goes above and below what one launch per rebuild
    is for, several times, with lists growing meanwhile: both captured graphs in
    turn, and still every member's run alone."""
    from openabl_amd import MEMBERS, Simulation, load_library, record_dtype
    from openabl_amd.ensemble import Ensemble, member_seed
    print("case ensemble rebuild forms in turn", flush=True)
    rng = np.random.default_rng(3)
    ms = [{"num_agents": int(n), "agent_density": 0.065536, "max_pos": fold6(math.sqrt(n / 0.065536)),
           "time_scale": 0.002} for n in rng.integers(300, 2000, 12)]
    cfg = {"hip.cell_scale": 1, "hip.tile": 1, "hip.nlist": 1}
    ens = Ensemble("boids2d", "f32", ms, config=cfg)
    ens.init(1, 2)
    forms = [ens.inspect("rebuild_launches")]
    for _ in range(90):
        ens.simulate(10)
        now = ens.inspect("rebuild_launches")
        if now != forms[-1]:
            forms.append(now)
    assert forms[:3] == [1, 4, 1]
    dt = record_dtype(MEMBERS["boids2d"], "f32")
    for m, p in enumerate(ms):
        load_library().abl_rng_seed(*member_seed(1, 2, m))
        sim = Simulation("boids2d", "f32", params=p, config=cfg)
        sim.init_agents()
        sim.simulate(900)
        assert field_bytes(ens.download(m)) == field_bytes(sim.download(dt)), m
        assert ens.inspect("list_capacity", m) == sim.inspect("list_capacity"), m
        sim.close()
    ens.close()
