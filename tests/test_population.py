"""Removal, birth, sorting and download kernels at the edges of their tiles.

  * predator_prey in index order against the oracle, bit for bit with ids, with
    populations around one birth tile (2,048), the limit of counting flags
    directly (32,768) and with more newborns than a block ranks at a time;
  * small populations sorted in one block equal the full sort
    (hip.grid=full), at 1 agent, the largest population and grid taken, and one
    beyond each.
"""
import numpy as np
import pytest

from orclib import Oracle, circle3d_params, circle_params, field_bytes, predator_prey_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prey", [255, 257, 2047, 2049, 33000])
def test_population_kernels_equal_oracle(prey):
    from openabl_amd import AGENTS, Simulation, load_library, record_dtype
    print(f"case population {prey} prey", flush=True)
    n = int(np.ceil(prey / 0.35))
    params = predator_prey_params(num_agents=n, REPRODUCE_PREY_PROB=0.3, REPRODUCE_PREDATOR_PROB=0.3)
    load_library().abl_rng_seed(0xDEADBEEF, 0xBEEFDEAD)
    sim = Simulation("predator_prey", "f64", params=params, config={"hip.order": "index"})
    sim.init_agents()
    o = Oracle("predator_prey").set(**params).init()
    for _ in range(3):
        sim.simulate(1)
        o.simulate(1)
        for t, (_, members) in enumerate(AGENTS["predator_prey"]):
            assert np.array_equal(sim.ids(t), o.ids(t)), t
            assert field_bytes(sim.download(record_dtype(members, "f64"), t)) == field_bytes(o.agents(t)), t
    assert len(o.agents(1)) > prey  # the populations grew past the tile
    sim.close()


@pytest.mark.parametrize("model,prec,params,cfg", [
    ("circle", "f64", circle_params(num_agents=1, rho=0.05, r=5.0), {}),
    ("circle", "f32", circle_params(num_agents=4096, rho=0.05, r=5.0), {"hip.cell_scale": 2}),
    ("circle", "f64", circle_params(num_agents=4097, rho=0.05, r=5.0), {}),
    # 8,000 and 9,261 cells: below and beyond the largest grid
    ("circle3d", "f64", circle3d_params(num_agents=3000, rho=3000 / 8e6, r=5.0), {"hip.cell_inflate": 1}),
    ("circle3d", "f32c", circle3d_params(num_agents=3000, rho=3000 / 9.2e6, r=5.0), {"hip.cell_inflate": 1}),
], ids=["one", "most-f32", "beyond", "3d", "3d-beyond"])
def test_small_sort_equals_full(model, prec, params, cfg):
    from openabl_amd import MEMBERS, Simulation, load_library, record_dtype
    print(f"case small sort {model} {prec} {params['num_agents']}", flush=True)
    out = []
    for grid in ("delta", "full"):
        load_library().abl_rng_seed(0xDEADBEEF, 0xBEEFDEAD)
        sim = Simulation(model, prec, params=params, config=dict(cfg, **{"hip.grid": grid}))
        sim.init_agents()
        sim.simulate(12)
        out.append((field_bytes(sim.download(record_dtype(MEMBERS[model], prec))), sim.neighbours(0)))
        sim.close()
    assert out[0][0] == out[1][0]
    assert all(np.array_equal(x, y) for x, y in zip(out[0][1], out[1][1]))


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_near_loops_reach_agents_at_nan(prec):
    """A near test accepts an agent whose position is NaN, and such agents are
    binned to an axis' first cells: the near loops narrowed to the radius still
    visit every one that the stencil holds (what index order does, whose sums
    are added in another order: 1e-4 and 1e-10 of a value or of 1 after one
    timestep, some 1,000 addends of 6e-8 and 1e-16)."""
    from openabl_amd import AGENTS, Simulation, record_dtype
    print(f"case population nan {prec}", flush=True)
    rng = np.random.default_rng(2)
    params = predator_prey_params(num_agents=6000)
    dts = [record_dtype(m, prec) for _, m in AGENTS["predator_prey"]]
    recs = [np.zeros(n, dt) for n, dt in zip((300, 2000, 3700), dts)]
    for rec in recs:
        rec["pos"] = rng.uniform(0, params["env_size"], rec["pos"].shape)
    for rec in recs[:2]:
        rec["dir"] = rng.uniform(-0.7, 0.7, rec["dir"].shape)
        rec["life"] = 40
        k = rng.choice(len(rec), 24, False)
        rec["pos"][k[:8], 0] = rec["pos"][k[8:16], 1] = rec["pos"][k[16:]] = np.nan
    outs = []
    for order in ("cell", "index"):
        sim = Simulation("predator_prey", prec, params=params, config={"hip.order": order})
        for t, rec in enumerate(recs):
            sim.upload(rec, t)
        sim.simulate(1)
        outs.append([sim.download(dt, t) for t, dt in enumerate(dts)])
        sim.close()
    tol = 1e-10 if prec == "f64" else 1e-4
    assert np.isnan(outs[0][1]["steer"]).any() and not np.isnan(outs[0][1]["steer"]).all()
    for a, b in zip(*outs):
        assert len(a) == len(b)
        for f in a.dtype.names:
            if a[f].dtype.kind == "f":
                assert np.array_equal(np.isnan(a[f]), np.isnan(b[f])), f
                assert np.allclose(a[f], b[f], rtol=tol, atol=tol, equal_nan=True), f
            else:
                assert np.array_equal(a[f], b[f]), f
