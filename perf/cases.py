"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values; "path" names the kind of work:

  steps     a resident run between two outputs: n F3D_time_steps (source, x and
            y sweeps in parity order, z sweep with deposition), then the
            concentration and the ground deposit read back into the arrays
            that the program keeps
  ensemble  the same for members of uneven sizes in batched launches
  meteo     one meteorological interval: corner fields to sweep fields, the CFL
            time step, the steps at that step, the read-back
  output    the result variables of one output time: concentration, surface
            concentration, column loads, cloud top, ground load, cuts
  stats     per-point statistics over the members of an ensemble
  train     Adam updates of the flux-correction network
  learned   steps of a coarse grid with the flux correction
  dropin    MODULE ADS's three sweeps called on host arrays, as FALL3D calls
            them

Read-backs go through the C entry fall3d_ads_get_state into page-locked
arrays allocated once, as a host program does that writes an output file at
every output time; outputs of a run with the FP32 states are single precision
(a host program of kind 4), those of the FP64 state double.

Fields are made on the GPU from the seed: winds of a few Fourier modes with
vertical shear (the operational generator's form), smooth diffusion
coefficients, log-spaced settling velocities growing with height, and clouds of
compact Gaussian puffs that fill a part of the domain.
"""
import ctypes
import math

import numpy as np
import torch

from fall3d_amd import ads

DEV = "cuda:0"
EPSILON = 1e-12  # Sources/mod_KindType.F90:42


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _steps(name, nx, ny, nz, nb, nsteps, state="fp32", limiter="minmod", marching="rk", stretched=False, stime=0.0,
           source=False, tune=False):
    return {"name": name, "path": "steps", "nx": nx, "ny": ny, "nz": nz, "nb": nb, "nsteps": nsteps, "state": state,
            "limiter": limiter, "marching": marching, "stretched": stretched, "stime": stime, "source": source,
            "tune": tune}


def listed():
    return [
        # a quick-look run: the 64x64x32 puff, where launches and latency are all there is
        _steps("puff_small_fp32", 64, 64, 32, 1, 100, source=True),
        # the operational domain with the default tile shapes and an erupting column
        _steps("operational_fp32", 360, 240, 60, 10, 40, source=True),
        # the large single domain (the benchmark's size, tuned as the benchmark tunes it), after the eruption
        _steps("large_fp32", 1024, 768, 80, 20, 40, tune=True),
        # a regional grid of odd sizes: compensated state, superbee, stretched levels, winds between two times
        _steps("regional_odd_fp32x2", 251, 187, 43, 7, 60, state="fp32x2", limiter="superbee", stretched=True,
               stime=0.35, source=True),
        # a truth run in the reference's double precision
        _steps("truth_fp64", 384, 288, 80, 12, 20, state="fp64"),
        # an uneven ensemble (the benchmark's ranges of member sizes), tuned as the benchmark tunes it
        {"name": "ensemble_uneven", "path": "ensemble", "members": 24, "nb": 6, "xy_min": 96, "xy_max": 256,
         "z_min": 40, "z_max": 60, "nsteps": 24, "sizes": 3},
        # one meteo interval of the operational domain: sigma levels over terrain, CMAQ, similarity, Ganser
        {"name": "meteo_interval", "path": "meteo", "nx": 360, "ny": 240, "nz": 60, "nb": 10, "map_v": 2, "modkh": 2,
         "modkv": 3, "modv": 2, "dry": True, "nsteps": 40},
        # one output time of the operational domain
        {"name": "output_products", "path": "output", "nx": 360, "ny": 240, "nz": 60, "nb": 10, "state": "fp32"},
        # probabilistic products of a 48-member ensemble on a 400x300 grid, four levels
        {"name": "ensemble_statistics", "path": "stats", "members": 48, "points": 480000},
        # training of the flux correction, batches as the benchmark takes them
        {"name": "network_training", "path": "train", "rows": 400000, "batch": 65536, "updates": 50},
        # the coarse run with the flux correction (half the benchmark's coarse domain in each horizontal direction,
        # half its bins)
        {"name": "learned_coarse", "path": "learned", "nx": 256, "ny": 192, "nz": 80, "nb": 10, "nsteps": 40},
        # FALL3D's own time loop calling MODULE ADS on its host arrays (single-precision build)
        {"name": "dropin_sweeps", "path": "dropin", "nx": 200, "ny": 150, "nz": 50, "nb": 8},
    ]


def _spread(rng, lo, hi):
    """An integer in lo..hi, uniform in the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps"] * 6 + ["ensemble", "meteo", "output", "stats", "train", "learned", "dropin"])
    if kind == "steps":
        state = rng.choice(["fp32", "fp32", "fp32x2", "fp64"])
        while True:
            nx, ny, nz, nb = _spread(rng, 24, 1024), _spread(rng, 20, 768), rng.randint(12, 90), _spread(rng, 1, 20)
            cells = nx * ny * nz * nb
            if 2e4 <= cells <= (6e7 if state == "fp64" else 4e8):
                break
        nsteps = 2 * rng.randint(5, 25 if cells > 1e8 else 40)
        return {k: v for k, v in _steps("", nx, ny, nz, nb, nsteps, state, rng.choice(["minmod", "minmod", "superbee", "ospre"]),
                                        rng.choice(["rk", "rk", "rk", "euler"]), rng.random() < 0.5,
                                        rng.choice([0.0, round(rng.uniform(0.05, 0.95), 2)]), rng.random() < 0.6,
                                        rng.random() < 0.3).items() if k != "name"}
    if kind == "ensemble":
        lo = rng.randint(40, 120)
        return {"path": "ensemble", "members": rng.randint(2, 24), "nb": rng.randint(1, 8), "xy_min": lo,
                "xy_max": lo + rng.randint(8, 130), "z_min": rng.randint(16, 40), "z_max": rng.randint(41, 64),
                "nsteps": 2 * rng.randint(5, 20), "sizes": rng.randint(0, 999)}
    if kind == "meteo":
        return {"path": "meteo", "nx": _spread(rng, 40, 420), "ny": _spread(rng, 40, 260), "nz": rng.randint(16, 62),
                "nb": rng.randint(2, 10), "map_v": rng.randint(0, 2), "modkh": rng.choice([1, 2, 4]),
                "modkv": rng.choice([1, 3]), "modv": rng.randint(1, 7), "dry": rng.random() < 0.5,
                "nsteps": 2 * rng.randint(5, 20)}
    if kind == "output":
        return {"path": "output", "nx": _spread(rng, 40, 420), "ny": _spread(rng, 40, 260), "nz": rng.randint(16, 62),
                "nb": rng.randint(2, 12), "state": rng.choice(["fp32", "fp32x2", "fp64"])}
    if kind == "stats":
        members = _spread(rng, 3, 200)
        return {"path": "stats", "members": members, "points": _spread(rng, 2000, 2000000 // max(members // 8, 1))}
    if kind == "train":
        return {"path": "train", "rows": _spread(rng, 20000, 400000), "batch": _spread(rng, 1000, 65536),
                "updates": rng.randint(5, 50)}
    if kind == "learned":
        return {"path": "learned", "nx": _spread(rng, 64, 300), "ny": _spread(rng, 64, 200), "nz": rng.randint(16, 80),
                "nb": rng.randint(2, 10), "nsteps": 2 * rng.randint(5, 20)}
    return {"path": "dropin", "nx": _spread(rng, 24, 260), "ny": _spread(rng, 24, 200), "nz": rng.randint(12, 60),
            "nb": rng.randint(1, 8)}


# ---------------------------------------------------------------------------
# inputs: arrays on the GPU, in the memory order of the reference's layouts
# (a Fortran array a(i, j, k) is a C-contiguous tensor [k, j, i] here)
# ---------------------------------------------------------------------------
DX, TOP = 5000.0, 20000.0  # horizontal spacing and domain top, m
DT = 20.0                  # time step of the resident runs, s: below the CFL limit of the winds below


def _levels(nz, stretched):
    """Corner levels 0..TOP: uniform, or spacing growing with height."""
    s = np.arange(nz + 1) / nz
    return TOP * ((0.6 * s + 0.4 * s * s) if stretched else s)


def _metrics(nx, ny, nz, stretched):
    """dX_p and dX_b of the three axes (Sources/mod_Grid.F90:485-562)."""
    z = _levels(nz, stretched)
    db = np.diff(z)
    zp = 0.5 * (z[1:] + z[:-1])
    dp = np.diff(zp)
    g = {"dX1_p": np.full(nx + 4, DX), "dX1_b": np.full(nx + 3, DX), "dX2_p": np.full(ny + 4, DX),
         "dX2_b": np.full(ny + 3, DX)}
    g["dX3_b"] = np.concatenate([db[:1], db, db[-1:], db[-1:]])
    g["dX3_p"] = np.concatenate([dp[:1], dp[:1], dp, dp[-1:], dp[-1:], dp[-1:]])
    return g


class _Weather:
    """Winds of random Fourier modes with shear, speeds up to about 15 m/s plus 2 m/s per km."""

    def __init__(self, seed):
        rng = np.random.default_rng(seed)
        n = 8
        lam = np.exp(rng.uniform(math.log(100e3), math.log(2000e3), n))
        ang = rng.uniform(0.0, 2.0 * math.pi, n)
        self.kx, self.ky = 2 * math.pi / lam * np.cos(ang), 2 * math.pi / lam * np.sin(ang)
        self.phase = rng.uniform(0.0, 2.0 * math.pi, n)
        self.rng = rng

    def _modes(self, x, y, weight):
        out = torch.zeros(y.numel(), x.numel(), dtype=torch.float64, device=DEV)
        for kx, ky, ph, w in zip(self.kx, self.ky, self.phase, weight):
            out += w * torch.cos(kx * x[None, :] + ky * y[:, None] + ph)
        return out * (15.0 / len(self.kx))

    def u(self, x, y):
        return self._modes(x, y, np.sign(self.ky))

    def v(self, x, y):
        return self._modes(x, y, -np.sign(self.kx))


def _axis(first, count, step):
    return (torch.arange(count, dtype=torch.float64, device=DEV) + first) * step


def _vset(nb):
    return 0.01 * 300.0 ** (np.arange(nb) / max(nb - 1, 1))


def _fields(c, seed, dtype):
    """Inputs of a resident run as GPU tensors: meteo in the argument order of set_meteo, grid, c, s."""
    nx, ny, nz, nb = c["nx"], c["ny"], c["nz"], c["nb"]
    stretched = c.get("stretched", False)
    z = torch.tensor(_levels(nz, stretched), device=DEV)
    zp = 0.5 * (z[1:] + z[:-1])
    zf = torch.cat([z[:1], z, z[-1:]])  # faces 0..nz+2
    wx = _Weather(seed)
    xf, yf, xc, yc = _axis(-1.0, nx + 3, DX), _axis(-1.0, ny + 3, DX), _axis(0.5, nx, DX), _axis(0.5, ny, DX)
    d = {}
    two = c.get("stime", 0.0) > 0.0
    for t in ("1", "2") if two else ("1",):
        late = 1.0 if t == "1" else 1.15
        d["u" + t] = (late * (wx.u(xf, yc)[None] + (2e-3 * zp)[:, None, None])).to(dtype)
        d["v" + t] = (late * wx.v(xc, yf).t()[None] + 0.0 * zp[:, None, None]).to(dtype)  # v(f, i, k): y fastest
        bell = torch.sin(math.pi * zf.clamp(0.0, TOP) / TOP)
        d["w" + t] = (late * 0.004 * wx.u(xc, yc)[:, :, None] * bell[None, None, :]).to(dtype)  # w(f, i, j)
    for a in "uvw":
        d.setdefault(a + "2", None)
    kh = 200.0 + 100.0 * torch.sin(2 * math.pi * torch.arange(nz, dtype=torch.float64, device=DEV) / nz)
    d["k1"] = kh[:, None, None].expand(nz, ny, nx + 4).to(dtype).contiguous()
    d["k2"] = kh[:, None, None].expand(nz, nx, ny + 4).to(dtype).contiguous()
    zk = torch.cat([zp[:1], zp[:1], zp, zp[-1:], zp[-1:]])
    k3 = 5.0 + 15.0 * torch.exp(-zk / 2000.0)
    d["k3"] = k3[None, None, :].expand(ny, nx, nz + 4).to(dtype).contiguous()
    vs = torch.tensor(_vset(nb), device=DEV)[:, None] * (1.0 + 0.5 * zf / TOP)[None, :]
    d["vs"] = vs[:, :, None, None].to(dtype).expand(nb, nz + 3, ny, nx).contiguous()
    d["grid"] = _metrics(nx, ny, nz, stretched)
    d["c"] = _cloud(wx.rng, nx, ny, nz, nb, z, dtype)
    d["s"] = None
    if c.get("source"):
        s = torch.zeros(nb, nz, ny, nx, dtype=dtype, device=DEV)
        col = zp < 12000.0
        i, j = int(wx.rng.integers(nx // 4, 3 * nx // 4)), int(wx.rng.integers(ny // 4, 3 * ny // 4))
        s[:, col, j, i] = 1e6 / (nb * max(int(col.sum()), 1))
        d["s"] = s
    return d


def _cloud(rng, nx, ny, nz, nb, z, dtype):
    """c(-1:nx+2, -1:ny+2, -1:nz+2, nb): four compact puffs of 1e-6 to 1e-3 kg/m3, exact zeros elsewhere."""
    x = torch.arange(-1, nx + 3, dtype=torch.float64, device=DEV)
    y = torch.arange(-1, ny + 3, dtype=torch.float64, device=DEV)
    zp = 0.5 * (z[1:] + z[:-1])
    zz = torch.cat([zp[:1], zp[:1], zp, zp[-1:], zp[-1:]]) / TOP
    out = torch.zeros(nb, nz + 4, ny + 4, nx + 4, dtype=dtype, device=DEV)
    for _ in range(4):
        cx, cy, cz = rng.uniform(0.2, 0.8) * nx, rng.uniform(0.2, 0.8) * ny, rng.uniform(0.2, 0.8)
        sx, sy, sz = rng.uniform(0.015, 0.05) * nx, rng.uniform(0.015, 0.05) * ny, rng.uniform(0.03, 0.10)
        peak = 10.0 ** rng.uniform(-6.0, -3.0)
        gx, gy, gz = (torch.exp(-0.5 * ((v - m) / w) ** 2) for v, m, w in ((x, cx, sx), (y, cy, sy), (zz, cz, sz)))
        p = peak * gz[:, None, None] * gy[None, :, None] * gx[None, None, :]
        p = torch.where(p > 1e-12, p, torch.zeros_like(p)).to(dtype)
        for b in range(nb):
            out[b] += p * (0.5 + 0.5 * b / nb)
    return out


def _host(t, pinned=True):
    """Host copy of a GPU tensor (page-locked, or as a Fortran program allocates it), as the Fortran-ordered array
    the API takes."""
    if t is None:
        return None
    h = torch.empty(t.shape, dtype=t.dtype, pin_memory=pinned)
    h.copy_(t)
    return h.numpy().T


def _dtype(state):
    return torch.float64 if state == "fp64" else torch.float32


def _context(c, d, state):
    g = ads.ADS(c["nx"], c["ny"], c["nz"], c["nb"], c.get("limiter", "minmod"), c.get("marching", "rk"),
                8 if state == "fp64" else 4, state, grid=d["grid"])
    _fill(g, d)
    return g


def _fill(g, d):
    if "u1" in d:
        g.set_meteo(*(_host(d[k]) for k in ("u1", "v1", "w1", "k1", "k2", "k3", "vs", "u2", "v2", "w2")))
    if d.get("s") is not None:
        g.set_source(_host(d["s"]))
    g.set_state(_host(d["c"]))


def _kept(nb, nx, ny, nz, dtype):
    """The arrays a program keeps for read-backs."""
    return {"c": torch.empty(nb, nz + 4, ny + 4, nx + 4, dtype=dtype, pin_memory=True),
            "acum": torch.empty(nb, ny + 4, nx + 4, dtype=dtype, pin_memory=True)}


def _read(g, out):
    rc = ads.load_library().fall3d_ads_get_state(g._h, ctypes.c_void_p(out["c"].data_ptr()),
                                                 ctypes.c_void_p(out["acum"].data_ptr()))
    if rc != 0:
        raise RuntimeError(f"fall3d_ads_get_state failed ({rc})")


# ---- ensemble ----------------------------------------------------------------
def _members(c):
    rng = np.random.default_rng(c["sizes"])
    n = c["members"]
    nx, ny = rng.integers(c["xy_min"], c["xy_max"] + 1, n), rng.integers(c["xy_min"], c["xy_max"] + 1, n)
    nz = rng.integers(c["z_min"], c["z_max"] + 1, n)
    return [{"nx": int(a), "ny": int(b), "nz": int(k), "nb": c["nb"], "source": True} for a, b, k in zip(nx, ny, nz)]


# ---- meteo ---------------------------------------------------------------------
def _corners(c, seed):
    """Corner fields at two times, grid factors and options of the meteo update, as host arrays."""
    nx, ny, nz, nb = c["nx"], c["ny"], c["nz"], c["nb"]
    wx = _Weather(seed)
    rng = wx.rng
    xc, yc = _axis(0.0, nx + 1, DX), _axis(0.0, ny + 1, DX)
    lev = torch.tensor(_levels(nz, False), device=DEV)
    hill = 400.0 + 300.0 * torch.sin(xc / (7.0 * DX))[None, :] * torch.cos(yc / (5.0 * DX))[:, None]
    h = hill if c["map_v"] else torch.zeros(ny + 1, nx + 1, dtype=torch.float64, device=DEV)
    z = h[None] + lev[:, None, None] * (1.0 - h / TOP)[None]
    gen = torch.Generator(device=DEV).manual_seed(int(seed))

    def noise(scale, shape):
        return scale * torch.randn(shape, generator=gen, dtype=torch.float64, device=DEV)

    def flat(lo, hi):
        return lo + (hi - lo) * torch.rand(ny + 1, nx + 1, generator=gen, dtype=torch.float64, device=DEV)

    corner = {k: [None, None] for k in ("uc", "vc", "wc", "tc", "tvc", "rhoc", "pblhc", "ustc", "monc")}
    for t in (0, 1):
        late = 1.0 + 0.15 * t
        tc = 288.0 + 2.0 * t - 6.5e-3 * z.clamp(max=11000.0) + noise(0.2, z.shape)
        vals = {"uc": late * (wx.u(xc, yc)[None] + 2e-3 * z) + noise(0.3, z.shape),
                "vc": late * wx.v(xc, yc)[None] + noise(0.3, z.shape), "wc": noise(0.05, z.shape), "tc": tc,
                "tvc": tc * 1.003, "rhoc": 1.225 * torch.exp(-z / 8500.0), "pblhc": flat(300.0, 1800.0),
                "ustc": flat(0.05, 0.6), "monc": flat(-400.0, 400.0)}
        for k, v in vals.items():
            corner[k][t] = _host(v.float(), pinned=False)
    corner["lusec"] = _host(flat(1.0, 24.9).floor().float())
    hp = 0.25 * (h[1:, 1:] + h[:-1, 1:] + h[1:, :-1] + h[:-1, :-1])
    mgrid = {"Hm1_p": np.ones(ny, np.float32), "Hm2_p": np.ones(ny + 4, np.float32),
             "Hm3_p": _host((1.0 - hp / TOP).float()), "dhdx_p": _host(((h[1:, 1:] - h[1:, :-1]) / DX).float()),
             "dhdy_p": _host(((h[1:, 1:] - h[:-1, 1:]) / DX).float()), "z_c": _host(z.float()), "h_c": _host(h.float()),
             "X3_c": lev.float().cpu().numpy(), "X3_p": (0.5 * (lev[1:] + lev[:-1])).float().cpu().numpy()}
    cat, agg = np.ones(nb, np.int32), np.zeros(nb, np.int32)
    if nb > 3:
        cat[0], agg[nb // 2] = 2, 1
    opts = {"map_h": 0, "map_v": c["map_v"], "modkh": c["modkh"], "modkv": c["modkv"], "modv": c["modv"], "kh0": 250.0,
            "kv0": 15.0, "rams_cs": 0.2275, "dlon": DX, "dlat": DX, "x3max": TOP, "s_time": 0.5, "vset_fac": 0.85,
            "diam": np.geomspace(2e-6, 1e-3, nb), "rho": rng.uniform(900.0, 2500.0, nb),
            "psi": rng.uniform(0.6, 0.99, nb), "cat": cat, "aggregate": agg, "dry_deposition": int(c["dry"])}
    return corner, mgrid, opts


# ---- output --------------------------------------------------------------------
def _output_inputs(c, seed):
    nx, ny, nz, nb = c["nx"], c["ny"], c["nz"], c["nb"]
    dtype = _dtype(c["state"])
    rng = np.random.default_rng(seed)
    lev = torch.tensor(_levels(nz, False), device=DEV)
    x, y = _axis(0.0, nx + 1, DX), _axis(0.0, ny + 1, DX)
    h = 400.0 + 300.0 * torch.sin(x / (7.0 * DX))[None, :] * torch.cos(y / (5.0 * DX))[:, None]
    z = (h[None] + lev[:, None, None] * (1.0 - h / TOP)[None]).to(dtype)
    acum = torch.rand(nb, ny + 4, nx + 4, generator=torch.Generator(device=DEV).manual_seed(int(seed)),
                      dtype=torch.float64, device=DEV)
    return {"c": _cloud(rng, nx, ny, nz, nb, lev, dtype), "acum": (0.01 * acum).to(dtype), "z": z,
            "hm3": (1.0 - 0.25 * (h[1:, 1:] + h[:-1, 1:] + h[1:, :-1] + h[:-1, :-1]) / TOP).to(dtype),
            "diam": np.geomspace(1e-6, 1e-3, nb), "pm": (10.0, 64.0), "sigma": np.arange(nz + 1) / nz,
            "x_cut": (0.31 * nx * DX, 0.62 * nx * DX), "y_cut": (0.43 * ny * DX,), "z_cut": (2000.0, 5000.0, 9000.0),
            "fl_cut": (50.0, 100.0, 200.0, 300.0)}


# ---- statistics, network ---------------------------------------------------------
PERCENTILES, THRESHOLDS = (5.0, 50.0, 75.0, 95.0), (1e-4, 1e-3, 2e-3, 1e-2)


def _member_fields(c, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    base = torch.randn(c["points"], generator=gen, dtype=torch.float64, device=DEV)
    spread = torch.randn(c["members"], c["points"], generator=gen, dtype=torch.float64, device=DEV)
    return 1e-3 * torch.exp(0.8 * base[None] + 0.6 * spread)


def _rows(c, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    x = torch.randn(c["rows"], 32, generator=gen, device=DEV).to(torch.bfloat16)
    w = torch.randn(32, generator=gen, device=DEV) / 6.0
    t = torch.tanh(x.float() @ w)
    return x.view(torch.int16).cpu().numpy().view(np.uint16), t.cpu().numpy()


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c, path = case, case["path"]
    if path == "steps":
        dtype = _dtype(c["state"])
        g = _context(c, _fields(c, seed, dtype), c["state"])
        if c["tune"] and c["state"] != "fp64":
            g.autotune(DT, c["stime"])
        return {"path": path, "case": c, "g": g, "out": _kept(c["nb"], c["nx"], c["ny"], c["nz"], dtype)}
    if path == "ensemble":
        ms = _members(c)
        e = ads.Ensemble([(m["nx"], m["ny"], m["nz"]) for m in ms], c["nb"], real_kind=4)
        n = sum(m["nb"] * (m["nx"] + 4) * (m["ny"] + 4) * (m["nz"] + 4) for m in ms)
        na = sum(m["nb"] * (m["nx"] + 4) * (m["ny"] + 4) for m in ms)
        flat = {"c": torch.empty(n, pin_memory=True), "acum": torch.empty(na, pin_memory=True)}
        parts, oc, oa = [], 0, 0
        for q, (m, g) in enumerate(zip(ms, e.members)):
            d = _fields(m, seed * 1000 + q, torch.float32)
            g.set_grid(d["grid"])
            _fill(g, d)
            lc = m["nb"] * (m["nx"] + 4) * (m["ny"] + 4) * (m["nz"] + 4)
            la = m["nb"] * (m["nx"] + 4) * (m["ny"] + 4)
            parts.append({"c": flat["c"][oc:oc + lc], "acum": flat["acum"][oa:oa + la]})
            oc, oa = oc + lc, oa + la
        e.autotune(DT)
        return {"path": path, "case": c, "e": e, "parts": parts, "out": flat}
    if path == "meteo":
        g = ads.ADS(c["nx"], c["ny"], c["nz"], c["nb"], real_kind=4,
                    grid=_metrics(c["nx"], c["ny"], c["nz"], False))
        lev = torch.tensor(_levels(c["nz"], False), device=DEV)
        g.set_state(_host(_cloud(np.random.default_rng(seed), c["nx"], c["ny"], c["nz"], c["nb"], lev, torch.float32)))
        return {"path": path, "case": c, "g": g, "corners": _corners(c, seed),
                "out": _kept(c["nb"], c["nx"], c["ny"], c["nz"], torch.float32)}
    if path == "output":
        d = _output_inputs(c, seed)
        g = ads.ADS(c["nx"], c["ny"], c["nz"], c["nb"], real_kind=8 if c["state"] == "fp64" else 4, state=c["state"],
                    grid=_metrics(c["nx"], c["ny"], c["nz"], False))
        g.set_state(_host(d["c"]), _host(d["acum"]))
        for k in ("z", "hm3"):
            d[k] = _host(d[k])
        return {"path": path, "case": c, "g": g, "d": d}
    if path == "stats":
        return {"path": path, "x": _member_fields(c, seed)}
    if path == "train":
        net = ads.Network(capacity=c["rows"], seed=seed)
        net.append(*_rows(c, seed))
        return {"path": path, "case": c, "net": net, "seed": seed}
    if path == "learned":
        g = _context(c, _fields(c, seed, torch.float32), "fp32")
        g.set_learned(ads.Network(seed=seed), smin=1e-10, gain=0.5)
        return {"path": path, "case": c, "g": g, "out": _kept(c["nb"], c["nx"], c["ny"], c["nz"], torch.float32)}
    d = _fields(c, seed, torch.float32)
    g = ads.ADS(c["nx"], c["ny"], c["nz"], c["nb"], real_kind=4, grid=d["grid"])
    h = {k: _host(d[k], pinned=False) for k in ("c", "k1", "k2", "k3", "w1", "vs")}
    u, v, _ = g.get_vcomps()
    u[...], v[...] = _host(d["u1"]), _host(d["v1"])
    h["acum"] = np.zeros(g.shape_acum, dtype=np.float32, order="F")
    return {"path": "dropin", "g": g, "h": h}


def run(state):
    path = state["path"]
    if path in ("steps", "learned"):
        c, g = state["case"], state["g"]
        g.run(DT, c["nsteps"], 0, c.get("stime", 0.0))
        _read(g, state["out"])
        return state["out"]
    if path == "ensemble":
        e = state["e"]
        e.run(DT, state["case"]["nsteps"])
        e.synchronize()
        for g, part in zip(e.members, state["parts"]):
            _read(g, part)
        return state["out"]
    if path == "meteo":
        g, c = state["g"], state["case"]
        g.update_meteo(*state["corners"])
        dt = g.time_step(0.5, 2, 0.9)
        g.run(dt, c["nsteps"], 0, 0.5)
        _read(g, state["out"])
        return {"dt": dt, **state["out"]}
    if path == "output":
        g, d = state["g"], state["d"]
        r = g.postprocess(z_c=d["z"], hm3=d["hm3"], pm_um=d["pm"], bin_diam=d["diam"],
                          want=("con", "con_sur", "col_mass", "col_mass_pm", "cloud_top", "grn_load", "grn_load_bin"))
        r.update(g.postprocess_cuts(d["z"], d["sigma"], TOP, dlon=DX, dlat=DX, x_cut=d["x_cut"], y_cut=d["y_cut"],
                                    z_cut=d["z_cut"], fl_cut=d["fl_cut"], hm3=d["hm3"]))
        return r
    if path == "stats":
        return ads.ensemble_statistics(state["x"], PERCENTILES, THRESHOLDS)
    if path == "train":
        c, net = state["case"], state["net"]
        loss = net.train(c["updates"], batch=c["batch"], lr=1e-3, seed=state["seed"])
        return {"loss": loss, "params": net.params()}
    g, h = state["g"], state["h"]
    f = [*g.solve_along_x(0.0, 0.0, DT, h["c"], h["k1"]), *g.solve_along_y(0.0, 0.0, DT, h["c"], h["k2"]),
         *g.solve_along_z(0.0, 0.0, DT, h["c"], h["acum"], h["k3"], h["w1"], h["w1"], 0.0, h["vs"])]
    return {"c": h["c"], "acum": h["acum"], "fluxes": np.array(f, dtype=np.float32)}


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _step_work(nx, ny, nz, nb, nsteps, state):
    """Bytes and operations of nsteps steps and the read-back: each sweep reads and writes the state once and
    reads its fields once; about 35 operations per cell, bin, stage and sweep (four stages)."""
    word, c = {"fp32": (4, 4), "fp32x2": (4, 8), "fp64": (8, 8)}[state]
    cells = nx * ny * nz
    back = (nx + 4) * (ny + 4) * (nz + 4) * nb * word
    return {"bytes": nsteps * cells * (nb * (6 * c + word) + 9 * word) + 2 * back, "flops": 420.0 * cells * nb * nsteps}


def work(case):
    c, path = case, case["path"]
    if path in ("steps", "learned", "meteo"):
        w = _step_work(c["nx"], c["ny"], c["nz"], c["nb"], c["nsteps"], c.get("state", "fp32"))
        if c.get("marching") == "euler":
            w["flops"] /= 4.0
        n = c["nx"] * c["ny"] * c["nz"]
        if path == "meteo":
            w["bytes"] += 4 * n * (12 + 9 + c["nb"])  # corner fields in, sweep fields out
            w["flops"] += n * (200.0 + 400.0 * c["nb"])
        if path == "learned":
            w["flops"] += 0.1 * 2 * n * c["nb"] * c["nsteps"] * 12400.0  # x and y faces of the cloud: a tenth of them
        return w
    if path == "ensemble":
        each = [_step_work(m["nx"], m["ny"], m["nz"], m["nb"], c["nsteps"], "fp32") for m in _members(c)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    if path == "output":
        n = c["nx"] * c["ny"] * c["nz"]
        state = {"fp32": 4, "fp32x2": 8, "fp64": 8}[c["state"]]
        return {"bytes": n * (2 * c["nb"] * state + 2 * 8 + 8 + 8), "flops": n * c["nb"] * 30.0}
    if path == "stats":
        n = c["points"]
        return {"bytes": 8.0 * n * (c["members"] + 4 + len(PERCENTILES) + len(THRESHOLDS)),
                "flops": n * c["members"] * (20.0 + 2.0 * math.log2(c["members"]) ** 2)}
    if path == "train":
        return {"bytes": c["updates"] * (c["batch"] * 68.0 + 6400 * 24.0), "flops": c["updates"] * c["batch"] * 37200.0}
    n = c["nx"] * c["ny"] * c["nz"]
    return {"bytes": n * (c["nb"] * (6 * 4 + 4) + 7 * 4.0), "flops": 420.0 * n * c["nb"]}


# ---------------------------------------------------------------------------
# exact: the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _slope(a, b, limiter):
    """phi(a/b) b of a cell with left difference a and right difference b (Sources/mod_ADS.F90:1124-1223)."""
    tiny = b.abs() < EPSILON
    r = a / torch.where(tiny, torch.ones_like(b), b)
    if limiter == "minmod":
        return torch.where(tiny, b, r.clamp_(0.0, 1.0).mul_(b))
    flat = a.abs() < EPSILON
    if limiter == "superbee":
        phi = torch.maximum(torch.clamp(2.0 * r, 0.0, 1.0), torch.clamp(r, 0.0, 2.0))
        edge = 2.0
    else:
        q = r * r + r
        phi = 1.5 * q / (q + 1.0)
        edge = 1.5
    return torch.where(tiny, torch.where(flat, torch.zeros_like(b), edge * b), phi * b)


def _sweep(c, axis, wind, kd, dxp, dxb, dt, limiter, marching):
    """One sweep of the lines c (all positions -1..n+2 along axis), in place; wind at faces 0..n+2, kd at
    positions -1..n+2. Returns |F + P| of the first face in the last stage."""
    n = c.shape[axis] - 4

    def cut(t, first, count):
        return t.narrow(axis, first, count)

    def along(v, first, count):
        shape = [1] * c.dim()
        shape[axis] = count
        return v[first:first + count].reshape(shape)

    u = cut(wind, 1, n + 1)
    kf = 0.5 * (cut(kd, 2, n + 1) + cut(kd, 1, n + 1)) / along(dxp, 1, n + 1)
    up, um = u.clamp(min=0.0), u.clamp(max=0.0)
    first, last = cut(c, 2, 1).clone(), cut(c, n + 1, 1).clone()
    gl = torch.where(cut(u, 0, 1) > 0.0, -first, first)
    gr = torch.where(cut(u, n, 1) < 0.0, -last, last)
    for p in (0, 1):
        cut(c, p, 1).copy_(gl)
        cut(c, n + 2 + p, 1).copy_(gr)
    width = along(dxb, 1, n)
    y, total, edge = c, None, None
    weights = (1.0,) if marching == "euler" else (1.0, 2.0, 2.0, 1.0)
    for st, wt in enumerate(weights):
        d = cut(y, 1, n + 3) - cut(y, 0, n + 3)                       # faces 0..n+2
        m = _slope(cut(d, 0, n + 2), cut(d, 1, n + 2), limiter)       # cells 0..n+1
        left = cut(y, 1, n + 1) + 0.5 * cut(m, 0, n + 1)
        right = cut(y, 2, n + 1) - 0.5 * cut(m, 1, n + 1)
        del m
        flux = left.mul_(up).add_(right.mul_(um))
        diff = kf * cut(d, 1, n + 1)
        del d, right
        if st == len(weights) - 1:
            edge = (cut(flux, 0, 1) + cut(diff, 0, 1)).abs()
        flux.sub_(diff)
        rhs = (cut(flux, 0, n) - cut(flux, 1, n)) / width
        total = rhs * wt if total is None else total.add_(rhs, alpha=wt)
        if st < len(weights) - 1:
            y = c.clone()
            cut(y, 2, n).add_(rhs, alpha=(0.5 if st < 2 else 1.0) * dt)
    cut(c, 2, n).add_(total, alpha=dt / sum(weights))
    return edge


def _exact_steps(case, d, nsteps):
    nx, ny, nz, nb = case["nx"], case["ny"], case["nz"], case["nb"]
    lim, tm, s = case.get("limiter", "minmod"), case.get("marching", "rk"), case.get("stime", 0.0)
    c, dt = d["c"].double(), DT
    acum = torch.zeros(nb, ny + 4, nx + 4, dtype=torch.float64, device=DEV)

    def at(a):
        t = d[a + "1"].double()
        return t if d.get(a + "2") is None else (1.0 - s) * t + s * d[a + "2"].double()

    u, v, w = at("u"), at("v").transpose(1, 2), at("w").permute(2, 0, 1)
    k1, k2, k3 = d["k1"].double(), d["k2"].double().transpose(1, 2), d["k3"].double().permute(2, 0, 1)
    word = d["c"].dtype  # the grid's spacings in the kind the program passes them
    g = {k: torch.tensor(a, device=DEV).to(word).double() for k, a in d["grid"].items()}
    src = None
    if d.get("s") is not None:
        vol = g["dX3_p"][2:nz + 2, None, None] * g["dX2_p"][None, 2:ny + 2, None] * g["dX1_p"][None, None, 2:nx + 2]
        src = dt * d["s"].double() / vol[None]
    inner = (slice(2, -2),) * 3
    for b in range(nb):
        weff = w - d["vs"][b].double()
        for it in range(nsteps):
            if src is not None:
                c[b][inner] += src[b]
            for axis in ((0, 1, 2) if it % 2 == 0 else (1, 0, 2)):
                if axis == 0:
                    _sweep(c[b][2:-2, 2:-2, :], 2, u, k1, g["dX1_p"], g["dX1_b"], dt, lim, tm)
                elif axis == 1:
                    _sweep(c[b][2:-2, :, 2:-2], 1, v, k2, g["dX2_p"], g["dX2_b"], dt, lim, tm)
                else:
                    e = _sweep(c[b][:, 2:-2, 2:-2], 0, weff, k3, g["dX3_p"], g["dX3_b"], dt, lim, tm)
                    acum[b][2:-2, 2:-2] += e[0] * dt
    return {"c": c, "acum": acum}


def _exact_output(d, c):
    nx, ny, nz, nb = c["nx"], c["ny"], c["nz"], c["nb"]
    z = d["z"].double()

    def clamped(t):  # a mass-point field with one more row on each side
        return torch.nn.functional.pad(t[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]

    hm3 = clamped(d["hm3"].double())
    con = torch.zeros(nz + 1, ny + 1, nx + 1, dtype=torch.float64, device=DEV)
    pm = torch.zeros(len(d["pm"]), nz + 1, ny + 1, nx + 1, dtype=torch.float64, device=DEV)
    grn = torch.zeros(nb, ny + 1, nx + 1, dtype=torch.float64, device=DEV)
    for b in range(nb):
        v = (1e3 * d["c"][b, 1:-1, 1:-1, 1:-1].double() / hm3[None]).clamp(min=0.0)
        v = 0.5 * (v[..., 1:] + v[..., :-1])
        v = 0.5 * (v[:, 1:] + v[:, :-1])
        v = 0.5 * (v[1:] + v[:-1])
        con += v
        for p, um in enumerate(d["pm"]):
            if d["diam"][b] <= um * 1e-6:
                pm[p] += v
        a = clamped(d["acum"][b, 2:-2, 2:-2].double())
        grn[b] = 0.25 * (a[1:, 1:] + a[:-1, 1:] + a[1:, :-1] + a[:-1, :-1])

    def load(t):
        return (0.5 * (t[1:] + t[:-1]) * (z[1:] - z[:-1])).sum(0)

    above = con > 50e-6
    top = torch.where(above, z, torch.full_like(z, -math.inf)).amax(0)
    top = torch.where(above.any(0), top, torch.zeros_like(top))
    levels = torch.tensor(d["sigma"] * TOP, device=DEV)

    def weights(x, at):  # interval and weight of the positions at among ascending x
        k = (torch.searchsorted(x, at) - 1).clamp(0, x.shape[-1] - 2)
        lo, hi = x.gather(-1, k), x.gather(-1, k + 1)
        return k, ((at - lo) / (hi - lo)).clamp(0.0, 1.0)

    cols, vals = z.permute(1, 2, 0).contiguous(), con.permute(1, 2, 0).contiguous()
    k, s = weights(cols, levels.expand(ny + 1, nx + 1, nz + 1).contiguous())
    cz = ((1.0 - s) * vals.gather(-1, k) + s * vals.gather(-1, k + 1)).permute(2, 0, 1)

    def cuts(x, at, dim):
        k, s = weights(x, torch.tensor(at, dtype=torch.float64, device=DEV))
        return [((1.0 - t) * cz.select(dim, int(q)) + t * cz.select(dim, int(q) + 1)) for q, t in zip(k, s)]

    xs, ys = _axis(0.0, nx + 1, DX), _axis(0.0, ny + 1, DX)
    out = {"con": con, "con_sur": con[0], "col_mass": load(con), "col_mass_pm": torch.stack([load(t) for t in pm]),
           "cloud_top": top, "grn_load": grn.sum(0), "grn_load_bin": grn,
           "cut_x": torch.stack(cuts(xs, d["x_cut"], 2)), "cut_y": torch.stack(cuts(ys, d["y_cut"], 1)),
           "cut_z": torch.stack(cuts(levels, d["z_cut"], 0)),
           "cut_fl": torch.stack(cuts(levels, [30.48 * f for f in d["fl_cut"]], 0))}
    # run() returns Fortran-ordered arrays: the reversed axes, in their order
    return {k: t.permute(*reversed(range(t.dim()))).contiguous() for k, t in out.items()}


def exact(case, seed):
    c, path = case, case["path"]
    if path == "steps":
        if 1.0 * c["nx"] * c["ny"] * c["nz"] * c["nb"] * c["nsteps"] > 6e9:
            return None  # minutes
        return _exact_steps(c, _fields(c, seed, _dtype(c["state"])), c["nsteps"])
    if path == "ensemble":
        ms = _members(c)
        if sum(1.0 * m["nx"] * m["ny"] * m["nz"] for m in ms) * c["nb"] * c["nsteps"] > 6e9:
            return None
        each = [_exact_steps(m, _fields(m, seed * 1000 + q, torch.float32), c["nsteps"]) for q, m in enumerate(ms)]
        return {k: torch.cat([e[k].reshape(-1) for e in each]) for k in ("c", "acum")}
    if path == "output":
        return _exact_output(_output_inputs(c, seed), c)
    if path == "stats":
        x = _member_fields(c, seed)
        n = x.shape[0]
        r = torch.sort(x, dim=0).values
        rank = [min(max(int(p / 100.0 * n), 1), n) - 1 for p in PERCENTILES]
        return {"mean": x.mean(0), "logmean": 10.0 ** torch.log10(x).mean(0), "stddev": x.std(0),
                "median": r[max(n // 2, 1) - 1], "per": r[rank],
                "prob": torch.stack([100.0 * (x >= t).double().sum(0) / n for t in THRESHOLDS])}
    if path == "dropin":
        d = _fields(c, seed, torch.float32)
        e = _exact_steps(c, d, 1)
        # run() returns Fortran-ordered arrays: the reversed axes, in their order
        return {**{k: t.permute(*reversed(range(t.dim()))).contiguous() for k, t in e.items()}, "fluxes": None}
    return None  # meteo, train, learned: iterative laws and a 16-bit network
