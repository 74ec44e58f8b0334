"""Source injection with map factors and grid changes of ensemble members,
through the C ABI on the GPU.

* set_source_metric divides by dX1_p dX2_p dX3_p Hm1_p(j) Hm2_p(j)
  Hm3_p(i,j) (Sources/mod_F3D.F90:1456-1473), checked against the FP64
  oracle's source add with the same factors over whole steps.
* A member whose grid changes between two runs at the same time step must
  be advanced with the new metrics: bit-identical to a single context set
  up with that grid.
"""
import numpy as np
import pytest

from fall3d_amd import ads
from fall3d_amd.problem import ensemble_members, random_problem, sigma_grid
from oracle.ads_oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("state", ["fp32", "fp32x2"])
def test_source_with_map_factors_matches_oracle(state):
    print(f"case: set_source_metric 20x16x10x2 state={state}", flush=True)
    p = random_problem(20, 16, 10, 2, seed=31)
    rng = np.random.default_rng(2)
    hm1 = rng.uniform(0.4, 1.0, p.ny)
    hm2 = np.ones(p.ny + 4)
    hm3 = rng.uniform(0.6, 1.0, (p.nx, p.ny))
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, state)
    g.set_problem(p)
    g.set_source(p.s, hm1=hm1, hm2=hm2, hm3=hm3)
    dt = 0.5 * g.time_step(0.0, 2, 0.9)
    g.run(dt, 3, 0)
    cg, ag = g.get_state()
    inj = g.budget()["injected"]
    g.release()
    o = Oracle(p, "minmod", "rk")
    c, acum = p.new_c(), p.new_acum()
    inj_o = 0.0
    for it in range(3):
        inj_o += o.add_source(dt, c, p.s, hm1=hm1, hm2=hm2, hm3=hm3)
        if it % 2 == 0:
            o.solve_x(dt, c, p.k1, p.u1)
            o.solve_y(dt, c, p.k2, p.v1)
        else:
            o.solve_y(dt, c, p.k2, p.v1)
            o.solve_x(dt, c, p.k1, p.u1)
        o.solve_z(dt, c, acum, p.k3, p.w1, p.w2, 0.0, p.vs)
    a, b = cg[2:-2, 2:-2, 2:-2], c[2:-2, 2:-2, 2:-2]
    err = np.linalg.norm(a - b) / np.linalg.norm(b)
    print(f"rel L2 {err:.3e}", flush=True)
    assert err <= 1e-5
    # with Hm = 1 the same source injects more mass: the factors are applied
    plain = Oracle(p, "minmod", "rk")
    c2 = p.new_c()
    assert plain.add_source(dt, c2, p.s) < inj_o
    # injected mass in the budget: dt s / (Hm1 Hm2 Hm3) in the dX_b measure of
    # this uniform grid. The compensated state adds the FP64 increment exactly;
    # the FP32 state records what its rounded cell values actually gained
    # (increments ~1e-4 of cell values of ~0.5 lose up to ~1e-3 of themselves)
    print(f"injected {inj!r} vs {inj_o!r}", flush=True)
    assert inj == pytest.approx(inj_o, rel=1e-12 if state == "fp32x2" else 1e-4)


def test_ensemble_member_grid_change_at_same_dt():
    print("case: ensemble member grid change", flush=True)
    specs = ensemble_members(3, nb=2, seed=5, nxy=(20, 60), nzr=(10, 14))
    ens = ads.Ensemble([(s.nx, s.ny, s.nz) for s in specs], 2, "minmod", "rk", 8, "fp32")
    probs = [sp.problem() for sp in specs]
    for gm, p in zip(ens.members, probs):
        gm.set_problem(p)
    dts = np.array([gm.time_step(0.0, 2, 0.9) for gm in ens.members]) * 0.25
    ens.run(dts, 2, 0)
    ens.synchronize()
    # member 1: new, stretched vertical grid; same dt, fresh state
    p1 = probs[1]
    s = np.concatenate([[0.0], np.cumsum(np.random.default_rng(4).uniform(0.5, 1.5, p1.nz))])
    g1 = sigma_grid(p1.nx, p1.ny, p1.nz, 5000.0, 5000.0, s / s[-1], p1.nz * 500.0)
    ens.members[1].set_grid(g1)
    ens.members[1].set_source(p1.s)  # the source is stored per unit volume of the grid
    ens.members[1].set_state(p1.c0)
    ens.members[1].set_fluxes(np.zeros(6))
    ens.run(dts, 3, 2)
    ens.synchronize()
    c_e, a_e = ens.members[1].get_state()
    tiling = ens.tiling()
    ens.release()
    p1.grid = g1
    g = ads.ADS(p1.nx, p1.ny, p1.nz, p1.nb, "minmod", "rk", 8, "fp32")
    g.set_problem(p1)
    g.set_tiling(0, cells_per_thread=tiling[0], bins_per_group=p1.nb)
    g.set_tiling(1, bins_per_group=tiling[1])
    g.set_tiling(2, bins_per_group=tiling[2])
    g.run(dts[1], 3, 2)
    c_s, a_s = g.get_state()
    g.release()
    assert np.all(np.isfinite(c_s))
    print(f"max |dc| {np.abs(c_e - c_s).max():.3e}", flush=True)
    assert np.array_equal(c_e, c_s)
    assert np.array_equal(a_e, a_s)


@pytest.mark.parametrize("kind,state", [(8, "fp64"), (4, "fp32")])
@pytest.mark.parametrize("nx", [2, 63, 64, 65, 130])
def test_sources_of_any_density(nx, kind, state):
    """set_source collects the entries of a row 64 at a time: rows that end
    before, at and after a piece, empty, with single values at a piece's ends,
    sparse and full, -0 among them. One step of the FP64 state equals the
    oracle's bit for bit, of the FP32 state within its tolerance. The injected
    mass of the FP32 state is what its cells took, c + inc rounded to FP32 (the
    increment too): 2^-24 of either per entry."""
    p = random_problem(nx, 7, 3, 2, seed=nx)
    rng = np.random.default_rng(nx)
    s = np.zeros_like(p.s)
    s[0, 1] = s[-1, 2] = 700.0
    s[min(63, nx - 1), 3] = s[min(64, nx - 1), 3, 1] = 900.0
    s[:, 4] = np.where(rng.random(s[:, 4].shape) < 0.1, 1e3 * rng.random(s[:, 4].shape), -0.0)
    s[:, 5] = 1e3 * rng.random(s[:, 5].shape)
    p.s[...] = s
    if kind == 4:
        p.s[...] = p.s.astype(np.float32)
    o = Oracle(p, 1, 2)
    dt = o.time_step(p.u1, p.v1, p.w1, p.vs, cfl=0.5)
    g = ads.ADS(nx, 7, 3, 2, 1, 2, kind, state)
    g.set_problem(p)
    c, acum = p.new_c(), p.new_acum()
    inj = o.step(dt, 0, c, acum)
    g.step(dt, 0)
    cg, _ = g.get_state()
    got = g.budget()["injected"]
    g.release()
    a, b = cg[2:-2, 2:-2, 2:-2].astype(np.float64), c[2:-2, 2:-2, 2:-2]
    if state == "fp64":
        assert np.array_equal(a, b)
    assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)
    meas = 1000.0 * 1200.0 * 150.0  # random_problem's uniform cells
    inc = dt * p.s / meas
    took = 0.0 if state == "fp64" else 2.0 ** -24 * meas * np.sum((np.abs(p.c0[2:-2, 2:-2, 2:-2]) + 2.0 * inc)[p.s != 0])
    assert abs(got - inj) <= 1e-12 * inj + took
