"""Parity of the gfx950 ADS kernels (through the C ABI) with the FP64 oracle.

Tolerances: the device computes reconstruction, fluxes and stage updates in
FP32 (FP64 only for the boundary/deposit accumulators, CFL and budget), so
concentrations and deposits are compared with relative L2 <= 1e-5 (the
required FP32 accuracy) and max-norm <= 1e-4 of the field's maximum; FP64-only
paths (ADS_solve_1D) with 1e-12. Mass conservation of the compensated
state (fp32x2) is checked to 1e-12 relative.
"""
import numpy as np
import pytest

from fall3d_amd import ads
from fall3d_amd.problem import operational_problem, puff_problem, random_problem
from oracle.ads_oracle import Oracle, solve_1d as ora_solve_1d, set_num_threads

pytestmark = pytest.mark.gpu

REL_L2 = 1e-5
MAX_REL = 1e-4


def rel_l2(a, b):
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (nb if nb > 0 else 1.0)


def check_field(gpu, ref, what, rel=REL_L2, mx=MAX_REL):
    e2 = rel_l2(gpu, ref)
    em = np.abs(gpu - ref).max() / max(np.abs(ref).max(), 1e-300)
    print(f"{what}: relL2={e2:.3e} max={em:.3e}", flush=True)
    assert e2 <= rel, (what, e2)
    assert em <= mx, (what, em)


def _dt(p, o, cfl=0.5):
    return o.time_step(p.u1, p.v1, p.w1, p.vs, criterion=2, cfl=cfl)


def _flux_scale(p, dt):
    vmax = max(np.abs(p.u1).max(), np.abs(p.v1).max(), np.abs(p.w1).max() + np.abs(p.vs).max())
    g = p.grid
    area = max(g["dX1_b"].max(), g["dX2_b"].max(), g["dX3_b"].max()) ** 2
    nl = max(p.nx * p.ny, p.ny * p.nz, p.nx * p.nz) * p.nb
    return vmax * np.abs(p.c0).max() * area * dt * nl


def _stretch_all_axes(p, seed):
    """Stretched metrics on every axis: a sigma grid in z (random_problem's
    stretched option, Sources/mod_Grid.F90:541-562) and independent random
    dX_p / dX_b arrays in x and y, so no two neighbouring cells share a
    spacing and dxp differs from dxb everywhere."""
    rng = np.random.default_rng(1000 + seed)
    g = p.grid
    for ax, n, d in ((1, p.nx, 1000.0), (2, p.ny, 1200.0)):
        g[f"dX{ax}_p"] = rng.uniform(0.6, 1.4, n + 4) * d
        g[f"dX{ax}_b"] = rng.uniform(0.6, 1.4, n + 3) * d
    return p


def _problem(seed, grid, *shape, **kw):
    if grid == "uniform":
        return random_problem(*shape, seed=seed, **kw)
    return _stretch_all_axes(random_problem(*shape, seed=seed, stretched=True, **kw), seed)


# ---------------------------------------------------------------------------
@pytest.mark.parametrize("grid", ["uniform", "stretched"])
@pytest.mark.parametrize("state", ["fp32", "fp32x2"])
@pytest.mark.parametrize("tm", [1, 2])
@pytest.mark.parametrize("lim", [1, 2, 3])
def test_dropin_sweeps_match_oracle(lim, tm, state, grid):
    """ADS_solve_along_x/y/z through the drop-in entry points, random problem
    (every face-velocity sign, ragged segment sizes, plateaus and zeros), on
    uniform and on stretched metrics of every axis."""
    print(f"case lim={lim} tm={tm} state={state} grid={grid}", flush=True)
    p = _problem(7 * lim + tm, grid, 13, 11, 9, 3)
    o = Oracle(p, lim, tm)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, lim, tm, 8, state, grid=p.grid)
    u, v, w = g.get_vcomps()
    u[...] = p.u1
    v[...] = p.v1
    dt = _dt(p, o)
    scale = _flux_scale(p, dt)
    cr, cg = p.new_c(), p.new_c()
    ar, ag = p.new_acum(), p.new_acum()
    o.solve_x(dt, cr, p.k1, p.u1)
    W, E = g.solve_along_x(0.0, 0.0, dt, cg, p.k1)
    check_field(cg, cr, "x sweep c")
    assert abs(W - o.flux[0]) <= 1e-5 * scale and abs(E - o.flux[1]) <= 1e-5 * scale
    o.solve_y(dt, cr, p.k2, p.v1)
    S, N = g.solve_along_y(0.0, 0.0, dt, cg, p.k2)
    check_field(cg, cr, "y sweep c")
    assert abs(S - o.flux[2]) <= 1e-5 * scale and abs(N - o.flux[3]) <= 1e-5 * scale
    o.solve_z(dt, cr, ar, p.k3, p.w1, p.w2, 0.3, p.vs)
    D, U = g.solve_along_z(0.0, 0.0, dt, cg, ag, p.k3, p.w1, p.w2, 0.3, p.vs)
    check_field(cg, cr, "z sweep c")
    check_field(ag, ar, "z sweep acum")
    assert abs(D - o.flux[4]) <= 1e-5 * scale and abs(U - o.flux[5]) <= 1e-5 * scale
    g.release()


def test_dropin_real4():
    """rp = 4 host kind (Sources/mod_KindType.F90:18-19, WITH_R4)."""
    p = random_problem(10, 9, 8, 2, seed=99)
    o = Oracle(p, 1, 2)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, 1, 2, 4, "fp32", grid=p.grid)
    u, v, w = g.get_vcomps()
    u[...] = p.u1.astype(np.float32)
    dt = _dt(p, o)
    cr = p.new_c()
    cg = np.asfortranarray(p.c0.astype(np.float32))
    o.solve_x(dt, cr, p.k1, np.asfortranarray(p.u1.astype(np.float32).astype(np.float64)))
    g.solve_along_x(0.0, 0.0, dt, cg, p.k1.astype(np.float32))
    check_field(cg.astype(np.float64), cr, "x sweep r4", rel=1e-5)


def test_update_horizontal_vcomps():
    p = random_problem(7, 6, 5, 1, seed=4)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, grid=p.grid)
    u2 = np.asfortranarray(p.u1 * 1.5 + 1.0)
    v2 = np.asfortranarray(p.v1 * 0.5 - 2.0)
    g.update_horizontal_vcomps(p.u1, u2, p.v1, v2, 0.25)
    u, v, _ = g.get_vcomps()
    np.testing.assert_allclose(u, 0.75 * p.u1 + 0.25 * u2, rtol=1e-6, atol=1e-6)
    np.testing.assert_allclose(v, 0.75 * p.v1 + 0.25 * v2, rtol=1e-6, atol=1e-6)


# ---------------------------------------------------------------------------
@pytest.mark.parametrize("grid", ["uniform", "stretched"])
@pytest.mark.parametrize("state", ["fp32", "fp32x2"])
def test_resident_steps_match_oracle(state, grid):
    """fall3d_ads_step = F3D_time_step (source, x/y order by parity, z) with
    time-interpolated winds (stime != 0), several steps, on uniform and
    stretched metrics."""
    print(f"case state={state} grid={grid}", flush=True)
    p = _problem(31, grid, 17, 12, 10, 2, umax_scale=0.5)
    o = Oracle(p, 1, 2)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, 1, 2, 8, state)
    g.set_problem(p)
    stime = 0.4
    u = np.asfortranarray((1 - stime) * p.u1 + stime * p.u2)
    v = np.asfortranarray((1 - stime) * p.v1 + stime * p.v2)
    w = np.asfortranarray((1 - stime) * p.w1 + stime * p.w2)
    dt = o.time_step(u, v, w, p.vs, cfl=0.5)
    dtg = g.time_step(stime=stime, criterion=2, cfl=0.5)
    assert dtg == pytest.approx(dt, rel=1e-6)
    cr, ar = p.new_c(), p.new_acum()
    for it in range(5):
        o.step(dt, it, cr, ar, stime=stime)
        g.step(dt, it, stime=stime)
    cg, ag = g.get_state()
    check_field(cg[2:-2, 2:-2, 2:-2], cr[2:-2, 2:-2, 2:-2], "resident c")
    check_field(ag, ar, "resident acum")
    fl = g.fluxes()
    scale = _flux_scale(p, dt) * 5
    assert np.all(np.abs(fl - o.flux) <= 1e-5 * scale), (fl, o.flux)


# ---------------------------------------------------------------------------
def test_puff_200_steps_matches_fp64():
    """64x64x32 Gaussian puff, one bin (v_s = 0.5 m/s), Kh = 100, Kv = 10,
    zero-flux laterals/top, absorbing ground, CFL 0.9, minmod + RK4, 200
    steps: FP32 device vs FP64 oracle (concentration and ground deposit)."""
    set_num_threads(16)
    p = puff_problem()
    o = Oracle(p, "minmod", "rk")
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32")
    g.set_problem(p)
    dt = o.time_step(p.u1, p.v1, p.w1, p.vs, cfl=0.9)
    dtg = g.time_step(0.0, 2, 0.9)
    assert dtg == pytest.approx(dt, rel=1e-6)
    cr, ar = p.new_c(), p.new_acum()
    for it in range(200):
        o.step(dt, it, cr, ar)
    g.run(dt, 200, 0)
    cg, ag = g.get_state()
    check_field(cg[2:-2, 2:-2, 2:-2], cr[2:-2, 2:-2, 2:-2], "puff c")
    check_field(ag, ar, "puff deposit")
    fl = g.fluxes()
    assert fl[4] == pytest.approx(o.flux[4], rel=1e-5)
    b = g.budget()
    assert b["mass_volume"] == pytest.approx(o.mass_volume(cr), rel=1e-5)


@pytest.mark.parametrize("state,tol", [("fp32x2", 1e-12)])
def test_puff_mass_conserved(state, tol):
    """Compensated state: domain mass + mass that left (ledger) = initial mass
    to FP64 rounding, over 200 steps."""
    p = puff_problem()
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, state)
    g.set_problem(p)
    dt = g.time_step(0.0, 2, 0.9)
    m0 = g.budget()["mass_cells"]
    g.run(dt, 200, 0)
    b = g.budget()
    err = abs(b["mass_cells"] + b["ledger"].sum() - m0) / m0
    print(f"mass closure {state}: {err:.3e} (deposited {b['ledger'][4] / m0:.3f} of M0)", flush=True)
    assert err <= tol


def test_operational_small_budget_closes():
    """Fourier wind with open laterals, 4 bins, line source: M + out = M0 + injected."""
    p = operational_problem(72, 48, 30, 4, seed=3)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32x2")
    g.set_problem(p)
    dt = g.time_step(0.0, 2, 0.9)
    g.run(dt, 60, 0)
    b = g.budget()
    assert b["injected"] > 0
    err = abs(b["mass_cells"] + b["ledger"].sum() - b["injected"]) / b["injected"]
    print(f"operational closure {err:.3e}", flush=True)
    assert err <= 1e-12


# ---------------------------------------------------------------------------
@pytest.mark.parametrize("lim", [1, 2, 3])
@pytest.mark.parametrize("bcode", [(2, 2), (1, 1), (-1, -1), (0, 2)])
def test_solve_1d_matches_oracle(lim, bcode):
    rng = np.random.default_rng(lim * 10 + bcode[0] + 5)
    n = 37
    c = rng.uniform(0.0, 1.0, n + 4)
    dxp = rng.uniform(500.0, 900.0, n + 4)
    dxb = rng.uniform(500.0, 900.0, n + 3)
    u = rng.normal(2.0, 3.0, n + 3)
    k = rng.uniform(10.0, 90.0, n + 4)
    cr = c.copy()
    fr = ora_solve_1d(cr, dxp, dxb, u, k, 20.0, (0.2, 0.7), bcode, lim)
    g = ads.ADS(4, 4, 4, 1)
    cg = c.copy()
    fg = g.solve_1d(cg, dxp, dxb, u, k, 20.0, (0.2, 0.7), bcode, 1, n, lim)
    np.testing.assert_allclose(cg, cr, rtol=1e-12, atol=1e-14)
    np.testing.assert_allclose(fg, fr, rtol=1e-11, atol=1e-14)


def test_deterministic_and_tiling_invariant():
    """Two runs are bitwise equal; other tilings (cells per lane of the x
    sweep, bins per workgroup) give the same concentration bits (shared faces
    are computed by the same instruction sequence); the FP64 ledger differs
    only by the summation order of the per-block partial sums."""
    p = operational_problem(40, 36, 20, 3, seed=5)
    outs = []
    for cpt, bpg in ((0, 0), (0, 0), (3, 1), (4, 2)):
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32x2")
        g.set_problem(p)
        if cpt or bpg:
            for ax in range(3):
                g.set_tiling(ax, cells_per_thread=cpt if ax == 0 else 0, bins_per_group=bpg)
        dt = g.time_step(0.0, 2, 0.9)
        g.run(dt, 6, 0)
        outs.append((g.get_state()[0], g.budget()["ledger"]))
        g.release()
    assert np.array_equal(outs[1][0], outs[0][0]) and np.array_equal(outs[1][1], outs[0][1])
    for c, led in outs[2:]:
        assert np.array_equal(c, outs[0][0])
        np.testing.assert_allclose(led, outs[0][1], rtol=1e-12, atol=1e-12 * np.abs(outs[0][1]).max())


@pytest.mark.parametrize("state,tm", [("fp32", "rk"), ("fp32x2", "rk"), ("fp32", "euler")])
def test_multiwave_x_lines_bit_identical(state, tm):
    """Lines held by 2 or 3 waves (edge cells traded through LDS) give the
    same bits as lines held by one wave."""
    p = operational_problem(200, 9, 6, 2, seed=8)
    outs = []
    for cpt in (4, 2, 3):  # 51 segments: one wave; 101 and 67: two waves
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", tm, 8, state)
        g.set_problem(p)
        g.set_tiling(0, cells_per_thread=cpt)
        dt = g.time_step(0.0, 2, 0.9)
        g.run(dt, 5, 0)
        outs.append(g.get_state())
        g.release()
    for c, a in outs[1:]:
        assert np.array_equal(c, outs[0][0])
        assert np.array_equal(a, outs[0][1])


def test_graph_replays_and_sampled_timing_match_direct_steps():
    """fall3d_ads_run with graph replays (from an even and an odd first
    iteration) and with per-kernel events on one step in 4 gives the same
    bits as direct launches; the sampled run times exactly the steps
    iiter0, iiter0 + 4, ..."""
    p = operational_problem(40, 36, 20, 3, seed=5)
    outs = []
    for mode in ("direct", "graph", "graph_odd", "sampled"):
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32")
        g.set_problem(p)
        dt = g.time_step(0.0, 2, 0.9)
        g.set_graph(mode != "direct")
        if mode == "graph_odd":
            g.run(dt, 5, 0)
            g.run(dt, 8, 5)
        else:
            g.set_profiling(4 if mode == "sampled" else 0)
            g.run(dt, 13, 0)
        if mode == "sampled":
            for k in ("sweep_x", "sweep_y", "sweep_z", "reduce"):
                ms, n = g.kernel_time(k)
                assert n == 4 and ms > 0.0, (k, n, ms)
            g.set_profiling(0)
        outs.append((g.get_state()[0], g.budget()["ledger"]))
        g.release()
    for c, led in outs[1:]:
        assert np.array_equal(c, outs[0][0])
        assert np.array_equal(led, outs[0][1])


@pytest.mark.parametrize("dims", [(40, 36, 20, 3), (70, 20, 3, 4), (33, 9, 2, 5), (65, 4, 2, 2)])
def test_stream_bins_per_thread_invariant(dims):
    """y/z streaming sweeps with two bins per thread give the concentration
    and deposit bits of one bin per thread (RK4 and Euler), also for lines
    shorter than the stage pipeline (nz = 2, 3), odd bin counts and
    partial 64-column tiles; the RK4 result matches the FP64 oracle."""
    print(f"case dims={dims}", flush=True)
    nx, ny, nz, nb = dims
    p = operational_problem(nx, ny, nz, nb, seed=sum(dims))
    for tm in ("rk", "euler"):
        outs = []
        for bpt in (1, 2):
            g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", tm, 8, "fp32")
            g.set_problem(p)
            for ax in (1, 2):
                g.set_tiling(ax, cells_per_thread=bpt, bins_per_group=2 if nb > 1 else 1)
            assert g.tiling(1)[0] == bpt and g.tiling(2)[0] == bpt
            dt = g.time_step(0.0, 2, 0.9)
            g.run(dt, 5, 0)
            outs.append((g.get_state(), g.budget()["ledger"], dt))
            g.release()
        (c1, a1), l1, dt = outs[0]
        (c2, a2), l2, _ = outs[1]
        assert np.array_equal(c1, c2) and np.array_equal(a1, a2), tm
        np.testing.assert_allclose(l2, l1, rtol=1e-12, atol=1e-12 * max(np.abs(l1).max(), 1e-300))
        if tm == "rk":
            o = Oracle(p, "minmod", "rk")
            cr, ar = p.new_c(), p.new_acum()
            for it in range(5):
                o.step(dt, it, cr, ar)
            check_field(c2[2:-2, 2:-2, 2:-2], cr[2:-2, 2:-2, 2:-2], f"c two bins per thread {dims}")


def test_operational_full_size_two_steps():
    """360x240x60, 10 bins (the benchmark workload) for two steps vs the
    FP64 oracle, plus budget closure of the compensated state."""
    set_num_threads(16)
    p = operational_problem()
    o = Oracle(p, "minmod", "rk")
    dt = o.time_step(p.u1, p.v1, p.w1, p.vs, cfl=0.9)
    cr, ar = p.new_c(), p.new_acum()
    for it in range(2):
        o.step(dt, it, cr, ar)
    for state in ("fp32", "fp32x2"):
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, state)
        g.set_problem(p)
        g.run(dt, 2, 0)
        cg, ag = g.get_state()
        check_field(cg[2:-2, 2:-2, 2:-2], cr[2:-2, 2:-2, 2:-2], f"operational c {state}")
        check_field(ag, ar, f"operational deposit {state}")
        if state == "fp32x2":
            b = g.budget()
            err = abs(b["mass_cells"] + b["ledger"].sum() - b["injected"]) / b["injected"]
            assert err <= 1e-12
        g.release()


@pytest.mark.parametrize("nx,cpt", [(12, 4), (12, 3), (13, 4), (16, 16), (64, 2), (63, 2), (40, 20),
                                    (128, 2), (200, 2), (383, 3), (300, 2), (500, 2), (1024, 6)])
def test_x_segmentation_edge_cases(nx, cpt):
    """x sweep with every segmentation case: cell n at the end of a segment
    (the last segment then holds only ghosts and face n+1), in its middle,
    one segment per line, and 64-lane lines; lines over 2, 3 and 4 waves
    (nx/cpt + 1 segments > 64), including a last wave whose only segment
    starts at face n+1; against the oracle."""
    print(f"case nx={nx} cpt={cpt}", flush=True)
    p = random_problem(nx, 7, 5, 2, seed=nx + cpt)
    o = Oracle(p, 1, 2)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, 1, 2, 8, "fp32", grid=p.grid)
    g.set_tiling(0, cells_per_thread=cpt)
    u, v, w = g.get_vcomps()
    u[...] = p.u1
    v[...] = p.v1
    dt = _dt(p, o)
    cr, cg = p.new_c(), p.new_c()
    o.solve_x(dt, cr, p.k1, p.u1)
    W, E = g.solve_along_x(0.0, 0.0, dt, cg, p.k1)
    check_field(cg, cr, "x sweep c")
    scale = _flux_scale(p, dt)
    assert abs(W - o.flux[0]) <= 1e-5 * scale and abs(E - o.flux[1]) <= 1e-5 * scale
    g.release()


# ---------------------------------------------------------------------------
@pytest.mark.parametrize("grid", ["uniform", "stretched"])
@pytest.mark.parametrize("stime", [0.0, 0.65])
def test_time_step_both_criteria(grid, stime):
    """grid_get_time_step (Sources/mod_Grid.F90:1026-1141) on the GPU with
    criterion 1 (largest per-direction rate) and criterion 2 (sum of the
    rates), for time-interpolated winds, against the FP64 oracle."""
    print(f"case grid={grid} stime={stime}", flush=True)
    p = _problem(44, grid, 23, 19, 11, 3)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32")
    g.set_problem(p)
    o = Oracle(p)
    u = np.asfortranarray((1 - stime) * p.u1 + stime * p.u2)
    v = np.asfortranarray((1 - stime) * p.v1 + stime * p.v2)
    w = np.asfortranarray((1 - stime) * p.w1 + stime * p.w2)
    for crit, cfl in ((1, 0.5), (2, 0.9)):
        ref = o.time_step(u, v, w, p.vs, criterion=crit, cfl=cfl)
        got = g.time_step(stime=stime, criterion=crit, cfl=cfl)
        print(f"criterion {crit}: {got!r} vs {ref!r}", flush=True)
        assert got == pytest.approx(ref, rel=1e-6)
    # the two criteria differ on this problem (the test tells them apart)
    assert o.time_step(u, v, w, p.vs, criterion=1, cfl=1.0) > 1.01 * o.time_step(u, v, w, p.vs, criterion=2, cfl=1.0)
    g.release()


def test_x_tiling_past_256_lanes_is_refused():
    """nx = 1024 at 3 or 4 cells per lane needs more than 256 lanes per x line:
    set_tiling returns an error and keeps the previous tiling."""
    g = ads.ADS(1024, 4, 4, 1)
    before = g.tiling(0)
    for cpt in (3, 4):
        with pytest.raises(ads.Fall3dAdsError, match="tiling"):
            g.set_tiling(0, cells_per_thread=cpt)
        assert g.tiling(0) == before
    g.release()


@pytest.mark.parametrize("case", ["puff", "operational", "stretched"])
def test_fp32_state_mass_closes_with_rounding_residual(case):
    """FP32 state: every final update is formed in FP64 and stored rounded to
    FP32; the mass that rounding moves is kept in the FP64 residual, so
    mass + ledger + residual - injected stays at the initial mass to FP64
    rounding (zero-flux puff, open operational domain with a source, and a
    problem stretched on every axis)."""
    if case == "puff":
        p, nsteps = puff_problem(), 200
    elif case == "operational":
        p, nsteps = operational_problem(72, 48, 30, 4, seed=3), 60
    else:
        p, nsteps = _problem(12, "stretched", 40, 33, 18, 3, umax_scale=0.5), 40
    print(f"case {case}", flush=True)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32")
    g.set_problem(p)
    dt = g.time_step(0.0, 2, 0.9 if case != "stretched" else 0.5)
    m0 = g.budget()["mass_cells"]
    g.run(dt, nsteps, 0)
    b = g.budget()
    g.release()
    ref = m0 + b["injected"]
    err = abs(b["mass_cells"] + b["ledger"].sum() + b["residual"] - ref) / ref
    naive = abs(b["mass_cells"] + b["ledger"].sum() - ref) / ref
    print(f"closure {err:.3e} (without the residual {naive:.3e}, residual {b['residual'] / ref:.3e})", flush=True)
    assert err <= 1e-12
    assert b["residual"] != 0.0


# ---------------------------------------------------------------------------
@pytest.mark.parametrize("dims", [(2, 2, 2, 1), (2, 5, 3, 2), (3, 2, 4, 3), (4, 3, 2, 2)])
@pytest.mark.parametrize("state", ["fp32", "fp64"])
def test_smallest_grids_match_oracle(dims, state):
    """The smallest grids the library accepts (2 cells along an axis): lines
    of 2-4 cells in every sweep, most cells next to a ghost. Resident steps
    with a source and time-interpolated winds against the oracle: the FP64
    state bit for bit, the FP32 state to the FP32 tolerances."""
    print(f"case dims={dims} state={state}", flush=True)
    p = random_problem(*dims, seed=sum(dims), umax_scale=0.5)
    o = Oracle(p, 1, 2)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, 1, 2, 8, state)
    g.set_problem(p)
    stime = 0.3
    u = np.asfortranarray((1 - stime) * p.u1 + stime * p.u2)
    v = np.asfortranarray((1 - stime) * p.v1 + stime * p.v2)
    w = np.asfortranarray((1 - stime) * p.w1 + stime * p.w2)
    dt = o.time_step(u, v, w, p.vs, cfl=0.5)
    cr, ar = p.new_c(), p.new_acum()
    for it in range(4):
        o.step(dt, it, cr, ar, stime=stime)
        g.step(dt, it, stime=stime)
    cg, ag = g.get_state()
    g.release()
    assert np.count_nonzero(cr[2:-2, 2:-2, 2:-2]) > 0
    if state == "fp64":
        assert np.array_equal(cg, cr) and np.array_equal(ag, ar)
    else:
        check_field(cg[2:-2, 2:-2, 2:-2], cr[2:-2, 2:-2, 2:-2], "smallest grid c")
        check_field(ag, ar, "smallest grid acum")


@pytest.mark.parametrize("dims,tm", [((64, 6, 5, 2), 2), ((65, 7, 4, 3), 2), ((130, 40, 26, 8), 2), ((33, 5, 200, 9), 2),
                                     ((20, 300, 7, 5), 1), ((190, 30, 12, 16), 2), ((251, 9, 6, 2), 2)])
def test_default_tile_shapes_match_oracle(dims, tm):
    """The tile shapes that a context picks by itself (cells per lane by the
    lanes a line fills, one or two bins per thread by how the waves fill the
    chip, odd bin counts included) give the oracle's field, also with
    face-flux output on, which runs the y sweep with one bin per thread."""
    print(f"case default tiles {dims} tm={tm}", flush=True)
    p = random_problem(*dims, seed=sum(dims))
    o = Oracle(p, 1, tm)
    dt = o.time_step(p.u1, p.v1, p.w1, p.vs, criterion=2, cfl=0.5)
    c, acum = p.new_c(), p.new_acum()
    for it in range(2):
        o.step(dt, it, c, acum)
    states = []
    for flux in ((False, True) if tm == 2 else (False,)):
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, 1, tm, 8, "fp32")
        g.set_problem(p)
        if flux:
            g.set_flux_output(True)
        for it in range(2):
            g.step(dt, it)
        print(f"  tiles {[g.tiling(d) for d in range(3)]}", flush=True)
        states.append(g.get_state())
        g.release()
        cg, ag = states[-1]
        a, b = cg[2:-2, 2:-2, 2:-2], c[2:-2, 2:-2, 2:-2]
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)
        assert np.linalg.norm(ag - acum) <= 1e-5 * np.linalg.norm(acum)
    if len(states) > 1:
        assert np.array_equal(states[0][0], states[1][0])


@pytest.mark.parametrize("state", ["fp32", "fp32x2"])
@pytest.mark.parametrize("lim,tm", [(1, 2), (2, 2), (3, 2), (1, 1)])
@pytest.mark.parametrize("dims", [(2, 3, 2, 1), (16, 4, 5, 3), (17, 7, 8, 2), (31, 127, 9, 2), (33, 128, 4, 1), (20, 255, 6, 2),
                                  (9, 256, 7, 5), (50, 503, 3, 1), (12, 504, 3, 1)])
def test_segmented_sweeps_equal_the_streaming_ones(dims, lim, tm, state):
    """Small grids run their y and z sweeps in segments by default; a tile
    shape set by hand runs the streaming kernels. Lines that end at every
    place of a segment, columns off the workgroup's, lines at the limits of
    the segment sizes (127/128, 255/256, 503/504 cells), bins over several
    workgroups, and the boundary rules: field, ghosts and deposit are equal
    bit for bit, the budget's sums to their rounding."""
    p = random_problem(*dims, seed=sum(dims), stretched=True)
    out = []
    for streaming in (False, True):
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, lim, tm, 8, state)
        g.set_problem(p)
        if streaming:
            for d in (1, 2):
                g.set_tiling(d, cells_per_thread=1, bins_per_group=1)
        dt = g.time_step(0.0, 2, 0.5)
        for it, bc in enumerate(("freeflow", "dirichlet", "periodic")):
            g.set_boundary(bc)
            g.step(dt, it, 0.25 * it)
        out.append((*g.get_state(), g.fluxes(), g.budget()))
        g.release()
    (c0, a0, f0, b0), (c1, a1, f1, b1) = out
    assert np.array_equal(c0, c1) and np.array_equal(a0, a1)
    scale = np.abs(f1).max() + abs(b1["mass_cells"])
    assert np.all(np.abs(f0 - f1) <= 1e-12 * scale)
    assert np.all(np.abs(b0["ledger"] - b1["ledger"]) <= 1e-12 * scale)
    assert abs(b0["residual"] - b1["residual"]) <= 1e-12 * scale


@pytest.mark.parametrize("state,lim,tm", [("fp32", 1, 2), ("fp32", 2, 2), ("fp32x2", 1, 2), ("fp32x2", 3, 1), ("fp32", 1, 1)])
@pytest.mark.parametrize("nx,nb", [(2, 3), (64, 1), (67, 5), (130, 2)])
def test_streaming_waves_and_line_ends(nx, nb, state, lim, tm):
    """The streaming sweeps' workgroups hold any number of consecutive waves,
    the last one fewer than its size, and the rows of a line arrive in groups
    of four that its ends cut anywhere: lines of 2 to 21 cells in y and z give
    the oracle's field in workgroups of 1, 3 and 8 waves of one bin and 1 and
    4 of two, all equal bit for bit."""
    for n in range(2, 22):
        p = random_problem(nx, n, 23 - n, nb, seed=100 * nx + n)
        o = Oracle(p, lim, tm)
        dt = o.time_step(p.u1, p.v1, p.w1, p.vs, criterion=2, cfl=0.5)
        c, acum = p.new_c(), p.new_acum()
        for it in range(2):
            o.step(dt, it, c, acum)
        ref = None
        for bpt, bpg in ((1, 1), (1, 3), (1, 8), (2, 2), (2, 8)):
            if bpt == 2 and state == "fp32x2":  # not a shape that can be set
                continue
            g = ads.ADS(p.nx, p.ny, p.nz, p.nb, lim, tm, 8, state)
            g.set_problem(p)
            for d in (1, 2):
                g.set_tiling(d, cells_per_thread=bpt, bins_per_group=bpg)
            for it in range(2):
                g.step(dt, it)
            cg, ag = g.get_state()
            g.release()
            if ref is None:
                ref = (cg, ag)
                a, b = cg[2:-2, 2:-2, 2:-2], c[2:-2, 2:-2, 2:-2]
                assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b), n
                assert np.linalg.norm(ag - acum) <= 1e-5 * np.linalg.norm(acum), n
            assert np.array_equal(cg, ref[0]) and np.array_equal(ag, ref[1]), (n, bpt, bpg)


@pytest.mark.parametrize("dims", [(64, 64, 32, 1), (64, 64, 32, 2), (40, 30, 20, 2), (360, 24, 60, 10), (200, 120, 50, 3)])
@pytest.mark.parametrize("state", ["fp32", "fp32x2"])
def test_reported_shapes_can_be_set_again(dims, state):
    """The shape that a context reports for an axis, set on it by hand, is the
    shape it had: bins per thread and waves of the streaming sweeps, and 0 for
    a y or z axis that runs in segments, which no explicit shape gives. The
    budget's sums follow the workgroups, so they are equal bit for bit. The
    same for the shapes that the autotuner reports."""
    p = random_problem(*dims, seed=sum(dims))
    print(f"case shapes {dims} {state}", flush=True)

    def run(tune=None, shapes=None):
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, 1, 2, 8, state)
        g.set_problem(p)
        dt = g.time_step(0.0, 2, 0.5)
        tuned = None
        if tune:
            tuned, _ = g.autotune(dt, 0.0, 1)
        if shapes:
            for d, (cpt, bpg) in enumerate(shapes):
                g.set_tiling(d, cells_per_thread=cpt, bins_per_group=bpg)
        for it in range(2):
            g.step(dt, it)
        got = [tuple(g.tiling(d)) for d in range(3)], g.budget(), g.get_state()[0]
        g.release()
        return (*got, tuned)

    for tune in (False, True):
        shapes, b0, c0, tuned = run(tune=tune)
        print(f"  {shapes} {tuned}", flush=True)
        if tune:
            assert list(tuned) == [shapes[0][0], shapes[1][1], shapes[2][1]]
        again, b1, c1, _ = run(shapes=shapes)
        assert again == shapes
        assert np.array_equal(c0, c1)
        for k in b0:
            assert np.array_equal(b0[k], b1[k]), k


def test_segments_return_after_face_fluxes():
    """Only the streaming y sweep writes face fluxes: a small grid leaves the
    segmented one while face-flux output is on, and has it back when that is
    off again, also if face fluxes were only needed for the learned limit."""
    p = random_problem(64, 64, 32, 1, seed=3)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, 1, 2, 8, "fp32")
    g.set_problem(p)
    before = [tuple(g.tiling(d)) for d in range(3)]
    g.set_flux_output(True)
    during = [tuple(g.tiling(d)) for d in range(3)]
    g.set_flux_output(False)
    after = [tuple(g.tiling(d)) for d in range(3)]
    net = ads.Network(params=ads.Network.initial_params(3))
    g.set_learned(net, smin=1e-12, gain=0.5, flux_limit=0.1)
    limited = [tuple(g.tiling(d)) for d in range(3)]
    g.set_learned(None)
    plain = [tuple(g.tiling(d)) for d in range(3)]
    g.release()
    assert before[1] == before[2] == (0, 0)
    assert during[1][1] > 0 and limited[1][1] > 0
    assert during[2] == limited[2] == (0, 0)
    assert after == plain == before


@pytest.mark.parametrize("axis", [1, 2])
@pytest.mark.parametrize("state,lim,tm", [("fp32", 1, 2), ("fp32", 2, 2), ("fp32x2", 3, 2), ("fp32x2", 1, 1), ("fp32", 3, 1)])
def test_segments_of_every_length_equal_the_stream(state, lim, tm, axis):
    """Lines that the automatic choice does run in segments (it reports 0 for
    them), ending at every cell of a segment: 4 cells per thread from the
    shortest such lines to 127 cells, 8 cells in 16 columns to 255 and in 8
    columns to 511. Field, ghosts and deposit equal the streaming kernel's bit
    for bit, fluxes and ledger to the rounding of their sums. 512 cells do not
    fit a workgroup and run in the stream."""
    shortest = 14 if axis == 1 else 6
    lengths = [*range(shortest, shortest + 5), 63, 126, 127, *range(128, 137), 255, *range(256, 265), 510, 511]
    for n in [*lengths, 512]:
        dims = (19, n, 3, 2) if axis == 1 else (19, 3, n, 2)
        p = random_problem(*dims, seed=n, stretched=True)
        out = []
        for streaming in (False, True):
            g = ads.ADS(p.nx, p.ny, p.nz, p.nb, lim, tm, 8, state)
            g.set_problem(p)
            if streaming:
                g.set_tiling(axis, cells_per_thread=1, bins_per_group=1)
            assert (g.tiling(axis)[1] == 0) == (not streaming and n < 512), n
            dt = g.time_step(0.0, 2, 0.5)
            for it, bc in enumerate(("freeflow", "dirichlet", "periodic")):
                g.set_boundary(bc)
                g.step(dt, it, 0.25 * it)
            out.append((*g.get_state(), g.fluxes(), g.budget()))
            g.release()
        (c0, a0, f0, b0), (c1, a1, f1, b1) = out
        assert np.array_equal(c0, c1) and np.array_equal(a0, a1), n
        scale = np.abs(f1).max() + abs(b1["mass_cells"])
        assert np.all(np.abs(f0 - f1) <= 1e-12 * scale), n
        assert np.all(np.abs(b0["ledger"] - b1["ledger"]) <= 1e-12 * scale), n
