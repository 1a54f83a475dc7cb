"""Timing cases of the LETKF analysis engine, through its public entry points.

Each case is one call as a user's program makes it: a single `letkf_core` from
a host loop, a batch of them on host arrays, one analysis cycle on device
arrays (obs index build, selection, products, transform, update) in each loop
the engine has, the whole `run_da` step (split, analysis, epilogue), the
observation operator, and a burst of jobs through the serving loop.  The
grids, ensemble sizes, obs counts, radii and options are those of the
configurations in `dida_letkf.synth`, `dida_letkf.serving`, `bench.py` and the
tests, with odd sizes between them.

Inputs: smooth random fields on the sphere (random plane waves whose
covariance has the length scale of a 500 km smoothing, correlated between
levels), evaluated exactly at the grid points and at the obs sites, so Yb has
the strongly correlated rows and A the steep spectrum that an ensemble gives.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dida-thhpca_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dida_letkf import engine  # noqa: E402
from dida_letkf.config import LetkfConfig  # noqa: E402

FP64, FP32, BF16X3 = 0, 1, 2
EARTH_KM = 6371.0
P0, PTOP = 1.0e5, 200.0
# real(4) constants of the distance and of the Gaspari-Cohn polynomial
PI_F = float(np.float32(np.arctan(np.float32(1.0)) * np.float32(4.0)))
A_F = float(np.float32(6371.393))
C1, C2 = float(np.float32(1.666667)), float(np.float32(0.6666667))


def _cycle(name, **kw):
    c = dict(kind="cycle", name=name, call="analyze", nlat=36, nlon=72, nz=1, n2d=1, n3d=0, k=20,
             n_obs=2000, mix="uniform", dist=1000.0, vert=0.0, lnp=False, halo=0, cube_n=1,
             cube_nz=1, overlap=0, prec=FP64, f32=False, rho=1.0, sigma=1.0)
    c.update(kw)
    return c


def listed():
    return [
        # the drop-in entry as the Fortran loop calls it, once per grid point: the
        # smallest call (a coarse ensemble with few local obs) ...
        dict(kind="core", name="core_one_k20", k=20, n=1, p=49, prec=FP64, rho=1.15),
        # ... and at the ensemble size and local obs count of the benchmarked cycle
        dict(kind="core", name="core_one_k64", k=64, n=1, p=1000, prec=FP64, rho=1.15),
        # many analyses from host arrays in one call, local obs counts ragged from 0
        dict(kind="core", name="core_batch_k40", k=40, n=256, p=400, prec=FP64, rho=1.1),
        # the smallest whole cycle: 72x36, one level and variable, 2,000 uniform obs
        _cycle("cycle_k20_72x36"),
        # the whole step of the driver (split, analysis, blended epilogue) on an odd
        # grid and ensemble, vertical localisation in ln p over chunks of 3 levels
        _cycle("run_da_lnp_k37_91x45", call="run_da", nlat=45, nlon=91, nz=8, n3d=3, k=37,
               n_obs=9001, mix="uniform3d", dist=800.0, vert=0.6, lnp=True, halo=1, cube_nz=3,
               rho=1.1),
        # overlapped cubes, the reference's default blocks (4 columns, overlap 2)
        _cycle("overlap_k20_96x48", nlat=48, nlon=96, nz=8, n3d=3, n_obs=20000,
               mix="uniform3d", dist=500.0, cube_n=4, overlap=2),
        # vertical loop at full size: one analysis per column and level (2 M solves)
        _cycle("vertical_k32_360x180", nlat=180, nlon=360, nz=32, n3d=3, k=32, n_obs=100_000,
               mix="uniform3d", dist=800.0, vert=2.0, prec=FP32, f32=True),
        # the benchmarked cycle: 500k clustered obs, split BF16 products, FP32 state
        _cycle("clustered_k64_360x180", nlat=180, nlon=360, nz=32, n3d=3, k=64, n_obs=500_000,
               mix="clustered", dist=300.0, prec=BF16X3, f32=True),
        # the same cycle in FP64 throughout
        _cycle("clustered_k64_360x180_fp64", nlat=180, nlon=360, nz=32, n3d=3, k=64,
               n_obs=500_000, mix="clustered", dist=300.0),
        # the largest ensemble on that grid
        _cycle("clustered_k128_360x180", nlat=180, nlon=360, nz=32, n3d=3, k=128,
               n_obs=500_000, mix="clustered", dist=300.0, prec=BF16X3, f32=True),
        # H(x) and its centring for a cycle's obs, before the analysis
        dict(kind="operator", name="operator_k64_360x180", nlat=180, nlon=360, nz=32, k=64,
             n_obs=200_000, stations=1000),
        # a burst of mixed jobs through the serving loop, three cycles each
        dict(kind="serve", name="serve_4_jobs", nlat=90, nlon=180, nz=16, ks="20,32,64,128",
             n_obs=60_000, prec=BF16X3),
    ]


def draw(rng):
    lg = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    what = rng.choice(["one", "batch", "cycle", "cycle", "clustered", "vertical", "run_da",
                       "overlap", "operator"])
    if what in ("one", "batch"):
        return dict(kind="core", k=lg(2, 128), n=1 if what == "one" else lg(2, 400),
                    p=lg(1, 2500 if what == "one" else 500),
                    prec=rng.choice([FP64, FP64, FP32, BF16X3]) if what == "batch" else FP64,
                    rho=round(rng.uniform(1.0, 1.3), 3))
    if what == "operator":
        nlat = rng.randint(20, 120)
        return dict(kind="operator", nlat=nlat, nlon=2 * nlat + rng.randint(0, 3),
                    nz=rng.randint(4, 24), k=lg(8, 128), n_obs=lg(500, 50_000),
                    stations=rng.randint(1, 200))
    nlat = lg(18, 130)
    nlon = 2 * nlat + rng.randint(-3, 3)
    prec = rng.choice([FP64, FP32, BF16X3])
    base = dict(nlat=nlat, nlon=nlon, nz=rng.randint(2, 24), n3d=rng.randint(1, 3), k=lg(8, 128),
                n_obs=lg(1000, 100_000), halo=rng.choice([0, 0, 1, 3]), prec=prec,
                rho=round(rng.uniform(1.0, 1.2), 3), sigma=round(math.exp(rng.uniform(-1.2, 1.1)), 3))
    if what == "cycle":
        c = _cycle("", mix="uniform3d", dist=float(rng.randint(250, 1000)),
                   f32=rng.random() < 0.4, **base)
    elif what == "clustered":
        c = _cycle("", mix="clustered", dist=float(rng.randint(200, 500)),
                   f32=rng.random() < 0.6, cube_n=rng.choice([1, 1, 2, 4]), **base)
    elif what == "run_da":
        c = _cycle("", call="run_da", mix="uniform3d", dist=float(rng.randint(250, 800)),
                   f32=rng.random() < 0.5, **base)
    elif what == "overlap":
        base.update(nlat=min(nlat, 60), nlon=min(nlon, 121), n_obs=min(base["n_obs"], 20000))
        cn = rng.randint(2, 5)
        c = _cycle("", mix="uniform3d", dist=float(rng.randint(250, 700)), cube_n=cn,
                   overlap=rng.randint(1, cn - 1), **base)
    else:
        base.update(nlat=min(nlat, 90), nlon=min(nlon, 181), k=lg(8, 80),
                    n_obs=min(base["n_obs"], 30_000))
        lnp = rng.random() < 0.5
        c = _cycle("", mix="uniform3d", dist=float(rng.randint(400, 900)),
                   vert=round(rng.uniform(0.3, 1.0) if lnp else rng.uniform(1.0, 3.0), 2),
                   lnp=lnp, cube_nz=rng.randint(1, 4), f32=rng.random() < 0.5, **base)
    c.pop("name")
    return c


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _xyz(lat, lon):
    la, lo = torch.deg2rad(lat), torch.deg2rad(lon)
    return torch.stack([torch.cos(la) * torch.cos(lo), torch.cos(la) * torch.sin(lo),
                        torch.sin(la)], dim=1)


class _Fields:
    """A truth and k members of n2d + n3d variables as sums of plane waves on
    the sphere; levels of a 3-D variable form an AR(1) sequence (0.8)."""
    WAVES = 192

    def __init__(self, k, nz, n2d, n3d, gen, dev):
        r = lambda *s: torch.randn(*s, generator=gen, device=dev, dtype=torch.float64)  # noqa: E731
        self.freq = r(3, self.WAVES) * (EARTH_KM / (math.sqrt(2.0) * 500.0))
        self.phase = torch.rand(self.WAVES, generator=gen, device=dev, dtype=torch.float64) * 2 * math.pi
        self.k, self.nz, self.n2d, self.n3d = k, nz, n2d, n3d
        self.coef = []                       # per state element: (WAVES, k + 1), truth last
        for v in range(n2d + n3d):
            prev = None
            for _ in range(1 if v < n2d else nz):
                c = r(self.WAVES, k + 1) * math.sqrt(2.0 / self.WAVES)
                c = c if prev is None else 0.8 * prev + 0.6 * c
                self.coef.append(c)
                prev = c

    def waves(self, lat, lon):
        return torch.cos(_xyz(lat, lon) @ self.freq + self.phase)

    def state(self, lat, lon, dtype):
        """xb (points, n, k) and axb (points, n) of the split state."""
        phi = self.waves(lat, lon)
        n = len(self.coef)
        xb = torch.empty((lat.numel(), n, self.k), dtype=dtype, device=lat.device)
        axb = torch.empty((lat.numel(), n), dtype=torch.float64, device=lat.device)
        for e, c in enumerate(self.coef):
            f = phi @ c
            m = f[:, :self.k].mean(dim=1)
            xb[:, e] = f[:, :self.k] - m[:, None]
            axb[:, e] = f[:, self.k] + m
        return xb, axb

    def rows(self, lat, lon, site, var, lev):
        """Centred members and (truth - mean) of H(x) at rows on `site`, of
        variable `var` at the (fractional, 1-based) level `lev`."""
        k = self.k
        phi = self.waves(lat, lon)
        start = torch.where(var < self.n2d, var, self.n2d + (var - self.n2d) * self.nz)
        l0 = torch.where(var < self.n2d, torch.zeros_like(var),
                         torch.clamp(lev.floor().long(), 1, max(self.nz - 1, 1)) - 1)
        wz = torch.where(var < self.n2d, torch.zeros_like(lev), lev - (l0 + 1))
        el = start + l0
        h = torch.empty((site.numel(), k + 1), dtype=torch.float64, device=lat.device)
        order = torch.argsort(el, stable=True)
        count = torch.bincount(el, minlength=len(self.coef)).tolist()
        at = 0
        for e, c in enumerate(count):
            if c == 0:
                continue
            idx = order[at:at + c]
            at += c
            up = self.coef[min(e + 1, len(self.coef) - 1)]
            f = phi[site[idx]]
            w = wz[idx][:, None]
            h[idx] = (1 - w) * (f @ self.coef[e]) + w * (f @ up)
        m = h[:, :k].mean(dim=1)
        return h[:, :k] - m[:, None], -m


def _sphere(rng, n):
    return np.rad2deg(np.arcsin(rng.uniform(-1.0, 1.0, n))), rng.uniform(0.0, 360.0, n)


def _swaths(rng, n, n_swaths=40, width_km=50.0):
    """Points on great circles, spread across a band around each."""
    plat, plon = _sphere(rng, n_swaths)
    which, t = rng.integers(0, n_swaths, n), rng.uniform(0.0, 2 * np.pi, n)
    off = rng.uniform(-0.5, 0.5, n) * width_km / EARTH_KM
    pl, po = np.deg2rad(plat)[which], np.deg2rad(plon)[which]
    p = np.stack([np.cos(pl) * np.cos(po), np.cos(pl) * np.sin(po), np.sin(pl)], 1)
    ref = np.where(np.abs(p[:, 2:]) < 0.9, [[0.0, 0.0, 1.0]], [[1.0, 0.0, 0.0]])
    e1 = np.cross(p, ref)
    e1 /= np.linalg.norm(e1, axis=1, keepdims=True)
    v = np.cos(off)[:, None] * (np.cos(t)[:, None] * e1 + np.sin(t)[:, None] * np.cross(p, e1)) \
        + np.sin(off)[:, None] * p
    return np.rad2deg(np.arcsin(np.clip(v[:, 2], -1, 1))), \
        np.mod(np.rad2deg(np.arctan2(v[:, 1], v[:, 0])), 360.0)


def _layout(mix, n_obs, nz, n2d, n3d, rng):
    """Site positions, rows per site, and variable and level of each row."""
    three = list(range(n2d, n2d + n3d)) or [0]
    if mix != "clustered":
        la, lo = _sphere(rng, n_obs)
        rp = np.arange(n_obs + 1)
        var = rng.choice(three, n_obs)
        return la, lo, rp, var, rng.uniform(1.0, max(float(nz), 1.000001), n_obs)
    # 70% on swaths, 20% in station columns (every level of every 3-D variable), 10% uniform
    per = nz * len(three)
    n_st = max(4, min(1000, n_obs // (5 * per)))
    n_sw = int(0.7 * n_obs)
    n_un = max(n_obs - n_sw - n_st * per, 0)
    a, b, c = _swaths(rng, n_sw), _sphere(rng, n_st), _sphere(rng, n_un)
    la, lo = np.concatenate([a[0], b[0], c[0]]), np.concatenate([a[1], b[1], c[1]])
    rows = np.concatenate([np.ones(n_sw, int), np.full(n_st, per), np.ones(n_un, int)])
    rp = np.concatenate([[0], np.cumsum(rows)])
    lev1 = lambda n: rng.uniform(1.0, max(float(nz), 1.000001), n)  # noqa: E731
    var = np.concatenate([rng.choice(three, n_sw), np.tile(np.tile(three, nz), n_st),
                          rng.choice(three, n_un)])
    lev = np.concatenate([lev1(n_sw), np.tile(np.repeat(np.arange(1.0, nz + 1), len(three)), n_st),
                          lev1(n_un)])
    return la, lo, rp, var, lev


def _t(a, dtype, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(dtype)


def _hybrid(nz):
    eta = np.linspace(0.0, 1.0, nz + 1)
    return eta - eta ** 2, eta ** 2


def _grid(nlat, nlon):
    return ((-90.0 + (np.arange(nlat) + 0.5) * 180.0 / nlat).astype(np.float32),
            ((np.arange(nlon) + 0.5) * 360.0 / nlon).astype(np.float32))


def _grid_points(glat, glon, dev):
    """Latitude and longitude of every column, longitude-major."""
    la, lo = _t(glat, torch.float64, dev), _t(glon, torch.float64, dev)
    return la.repeat(lo.numel()), lo.repeat_interleave(la.numel())


def _obs_set(fld, mix, n_obs, sigma, rng, gen, dev, lnp=False):
    la, lo, rp, var, lev = _layout(mix, n_obs, fld.nz, fld.n2d, fld.n3d, rng)
    site = np.repeat(np.arange(la.size), np.diff(rp))
    o = dict(lat=_t(la, torch.float64, dev), lon=_t(lo, torch.float64, dev),
             rp=_t(rp, torch.int32, dev), site=_t(site, torch.int64, dev))
    tv, tl = _t(var, torch.int64, dev), _t(lev, torch.float64, dev)
    yb, dep = fld.rows(o["lat"], o["lon"], o["site"], tv, tl)
    # error 1 for the last variable (temperature), 2 for the others, times sigma
    s = torch.where(tv == fld.n2d + fld.n3d - 1, 1.0, 2.0).double() * sigma
    o["yb"] = yb.contiguous()
    o["dep"] = dep + s * torch.randn(s.numel(), generator=gen, device=dev, dtype=torch.float64)
    o["rinv"] = 1.0 / (s * s)
    if lnp:      # ln p of the level in a standard atmosphere
        hya, hyb = _hybrid(fld.nz)
        ph = hya * (P0 - PTOP) + hyb * (P0 - PTOP) + PTOP
        mid = np.log(0.5 * (ph[:-1] + ph[1:]))
        tl = _t(np.interp(lev, np.arange(1, fld.nz + 1), mid), torch.float64, dev)
    o["vco"] = tl
    o["n_sites"], o["n_rows"] = la.size, int(rp[-1])
    return o


def _with_halo(a, nlon, nlat, h):
    """[nlon * nlat, ...] columns into [nlon + 2h, nlat + 2h, ...]: periodic in
    longitude, the nearest row past either pole."""
    a = a.reshape(nlon, nlat, *a.shape[1:])
    if h == 0:
        return a.contiguous()
    i = torch.arange(-h, nlon + h, device=a.device) % nlon
    j = torch.clamp(torch.arange(-h, nlat + h, device=a.device), 0, nlat - 1)
    return a[i][:, j].contiguous()


def _config(c):
    cfg = LetkfConfig(k=c["k"], nlat=c["nlat"], nlon=c["nlon"], nz=c["nz"], n2d=c["n2d"],
                      n3d=c["n3d"], halo=c["halo"], local_dist=c["dist"],
                      vert_dist=c["vert"] if c["vert"] > 0 else -1.0, inflation_factor=c["rho"],
                      cube_n=c["cube_n"], cube_nz=c["cube_nz"], overlap=c["overlap"],
                      precision=c["prec"], vcoord_mode=1 if c["lnp"] else 0)
    if c["lnp"]:
        hya, hyb = _hybrid(c["nz"])
        cfg.hyai, cfg.hybi, cfg.p0, cfg.ptop = list(hya), list(hyb), P0, PTOP
    return cfg


def _cycle_inputs(c, seed):
    dev = _dev()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 7919 + 11)
    rng = np.random.Generator(np.random.Philox(seed * 7919 + 12))
    fld = _Fields(c["k"], c["nz"], c["n2d"], c["n3d"], gen, dev)
    glat, glon = _grid(c["nlat"], c["nlon"])
    full = c["call"] == "run_da"
    f32 = c["f32"] and not full
    xb, axb = fld.state(*_grid_points(glat, glon, dev), torch.float32 if f32 else torch.float64)
    obs = _obs_set(fld, c["mix"], c["n_obs"], c["sigma"], rng, gen, dev, c["lnp"])
    if c["lnp"]:                       # surface pressure in Pa: 1e5, spread 300
        axb[:, 0] = 1.0e5 + 1000.0 * axb[:, 0]
        xb[:, 0] *= 300.0
    h = c["halo"]
    xb, axb = _with_halo(xb, c["nlon"], c["nlat"], h), _with_halo(axb, c["nlon"], c["nlat"], h)
    return xb, axb, obs, glat, glon


def _core_inputs(c, seed):
    rng = np.random.Generator(np.random.Philox(seed * 7919 + 13))
    k, out = c["k"], []
    # ragged counts, 0 and p among them
    ps = [c["p"]] if c["n"] == 1 else [0, c["p"]] + list(rng.integers(0, c["p"] + 1, c["n"] - 2))
    mem = rng.standard_normal((k, 40))
    for p in ps:
        # rows of correlated obs: 40 common modes with a falling spectrum, plus noise
        load = rng.standard_normal((40, p)) * np.exp(-0.15 * np.arange(40))[:, None]
        y = mem @ load * 0.4 + 0.3 * rng.standard_normal((k, p))
        y = np.asfortranarray(y - y.mean(axis=0, keepdims=True))
        out.append((y, (1.0 / rng.uniform(0.5, 2.0, p) ** 2).astype(np.float32),
                    rng.standard_normal(p), rng.uniform(0.0, 1.0, p)))
    return out


def _operator_inputs(c, seed):
    dev = _dev()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 7919 + 14)
    rng = np.random.Generator(np.random.Philox(seed * 7919 + 15))
    nz, n = c["nz"], 1 + 3 * c["nz"]
    fld = _Fields(c["k"], nz, 1, 3, gen, dev)
    glat, glon = _grid(c["nlat"], c["nlon"])
    xb, axb = fld.state(*_grid_points(glat, glon, dev), torch.float64)
    axb[:, 0] = 1.0e5 + 1000.0 * axb[:, 0]
    xb[:, 0] *= 300.0
    xb, axb = _with_halo(xb, c["nlon"], c["nlat"], 1), _with_halo(axb, c["nlon"], c["nlat"], 1)
    # single-level obs, surface-pressure obs (1 in 20) and sounding columns
    la, lo = _sphere(rng, c["n_obs"] + c["stations"])
    one = rng.uniform(np.log(2 * PTOP), np.log(1.05e5), c["n_obs"])
    var1 = np.where(rng.random(c["n_obs"]) < 0.05, 0, rng.integers(1, 4, c["n_obs"]))
    prof = np.sort(rng.uniform(np.log(1000.0), np.log(1.0e5), (c["stations"], nz)), axis=1)
    rows = np.concatenate([np.ones(c["n_obs"], int), np.full(c["stations"], 3 * nz)])
    rp = np.concatenate([[0], np.cumsum(rows)])
    o = dict(lat=_t(la, torch.float64, dev), lon=_t(lo, torch.float64, dev),
             rp=_t(rp, torch.int32, dev), n_sites=la.size, n_rows=int(rp[-1]),
             site=_t(np.repeat(np.arange(la.size), rows), torch.int64, dev),
             var=_t(np.concatenate([var1, np.tile([1, 2, 3], c["stations"] * nz)]), torch.int32, dev),
             ph=_t(np.exp(np.concatenate([one, np.repeat(prof.reshape(-1), 3)])), torch.float64, dev))
    o["yo"] = torch.randn(o["n_rows"], generator=gen, device=dev, dtype=torch.float64)
    return xb, axb, o, glat, glon, n


def _serve_jobs(c, seed):
    dev = _dev()
    jobs = []
    for j, k in enumerate(int(s) for s in c["ks"].split(",")):
        cc = _cycle("", nlat=c["nlat"], nlon=c["nlon"], nz=c["nz"], n3d=3, k=k, mix="clustered",
                    n_obs=c["n_obs"], dist=300.0, prec=c["prec"])
        gen = torch.Generator(device=dev)
        gen.manual_seed(seed * 7919 + 20 + j)
        rng = np.random.Generator(np.random.Philox(seed * 7919 + 30 + j))
        fld = _Fields(k, c["nz"], 1, 3, gen, dev)
        glat, glon = _grid(c["nlat"], c["nlon"])
        xb, axb = fld.state(*_grid_points(glat, glon, dev), torch.float64)
        xb = _with_halo(xb, c["nlon"], c["nlat"], 0)
        axb = _with_halo(axb, c["nlon"], c["nlat"], 0)
        cycles = [_obs_set(fld, "clustered", c["n_obs"], 1.0, rng, gen, dev) for _ in range(3)]
        jobs.append(dict(case=cc, cfg=_config(cc), xb=xb, axb=axb, obs=cycles, glat=glat, glon=glon,
                         xa=torch.zeros_like(xb), axa=torch.zeros_like(axb)))
    return jobs


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "core":
        return dict(c=c, inputs=_core_inputs(c, seed))
    if c["kind"] == "serve":
        s = dict(c=c, jobs=_serve_jobs(c, seed))
        s["server"] = engine.Server(24 << 30, max_active=4)
        torch.cuda.synchronize()
        return s
    if c["kind"] == "operator":
        xb, axb, o, glat, glon, n = _operator_inputs(c, seed)
        hya, hyb = _hybrid(c["nz"])
        cfg = LetkfConfig(k=c["k"], nlat=c["nlat"], nlon=c["nlon"], nz=c["nz"], n2d=1, n3d=3,
                          halo=1, hyai=list(hya), hybi=list(hyb), p0=P0, ptop=PTOP)
        s = dict(c=c, xb=xb, axb=axb, o=o,
                 yb=torch.empty((o["n_rows"], c["k"]), dtype=torch.float64, device=xb.device),
                 dep=torch.empty(o["n_rows"], dtype=torch.float64, device=xb.device))
    else:
        cfg = _config(c)
        xb, axb, o, glat, glon = _cycle_inputs(c, seed)
        s = dict(c=c, o=o)
        if c["call"] == "run_da":
            s["x_in"] = xb + axb[..., None]
            shape = (c["nlon"], c["nlat"], cfg.n)
            s["out"] = [torch.zeros_like(xb)] + [torch.zeros(shape, dtype=torch.float64,
                                                             device=xb.device) for _ in range(2)]
        else:
            s.update(xb=xb, axb=axb, xa=torch.zeros_like(xb), axa=torch.zeros_like(axb))
    eng = engine.LetkfEngine(cfg)
    eng.set_stream(torch.cuda.current_stream().cuda_stream)
    eng.set_grid(glat, glon)
    s["eng"] = eng
    torch.cuda.synchronize()
    return s


POLAR, GAMMA1, GAMMA2 = 85.0, 0.2, 0.8


def run(s):
    c = s["c"]
    if c["kind"] == "core":
        x = s["inputs"]
        if c["n"] == 1:
            return engine.letkf_core(*x[0], inflation_factor=c["rho"])
        return engine.letkf_core_batched([v[0] for v in x], [v[1] for v in x], [v[2] for v in x],
                                         [v[3] for v in x], inflation_factor=c["rho"],
                                         precision=c["prec"])
    if c["kind"] == "serve":
        srv, ids = s["server"], []
        for j in s["jobs"]:
            cyc = [dict(n_sites=o["n_sites"], n_rows=o["n_rows"], site_lat=o["lat"].data_ptr(),
                        site_lon=o["lon"].data_ptr(), site_row_ptr=o["rp"].data_ptr(),
                        yb=o["yb"].data_ptr(), dep=o["dep"].data_ptr(), rinv=o["rinv"].data_ptr(),
                        vcoord=o["vco"].data_ptr()) for o in j["obs"]]
            ids.append(srv.submit(j["cfg"], j["glat"], j["glon"], j["xb"].data_ptr(),
                                  j["axb"].data_ptr(), cyc, j["xa"].data_ptr(),
                                  j["axa"].data_ptr()))
        rcs = [srv.wait(i) for i in ids]
        return [[r["rc"] for r in rcs]] + [[j["xa"], j["axa"]] for j in s["jobs"]]
    o, eng = s["o"], s["eng"]
    if c["kind"] == "operator":
        eng.obs_operator_device(s["xb"].data_ptr(), s["axb"].data_ptr(), o["n_sites"],
                                o["lat"].data_ptr(), o["lon"].data_ptr(), o["rp"].data_ptr(),
                                o["n_rows"], o["var"].data_ptr(), o["ph"].data_ptr(),
                                o["yo"].data_ptr(), s["yb"].data_ptr(), s["dep"].data_ptr())
        return [s["yb"], s["dep"]]
    eng.set_obs_device(o["n_sites"], o["lat"].data_ptr(), o["lon"].data_ptr(), o["rp"].data_ptr(),
                       o["n_rows"], o["yb"].data_ptr(), o["dep"].data_ptr(), o["rinv"].data_ptr(),
                       o["vco"].data_ptr())
    if c["call"] == "run_da":
        out = s["out"]
        rc = eng.run_da_device(s["x_in"].data_ptr(), POLAR, GAMMA1, GAMMA2, out[0].data_ptr(),
                               out[1].data_ptr(), out[2].data_ptr(), state_f32=c["f32"])
        return [rc] + out
    f = eng.analyze_device_f32 if c["f32"] else eng.analyze_device
    rc = f(s["xb"].data_ptr(), s["axb"].data_ptr(), s["xa"].data_ptr(), s["axa"].data_ptr())
    return [rc, s["xa"], s["axa"]]


# --------------------------------------------------------------------------
# the work a pass cannot do without
# --------------------------------------------------------------------------

def _cycle_work(c, state_bytes):
    """Expected over uniform site positions.  Per analysis with p local rows:
    the symmetric product k(k+1)p and Yb^T R^-1 d 2kp, the inverse square root
    of a k x k matrix 4/3 k^3 (reduction) + 2 k^3, overline_w 4k^2; per state
    row of the column 2k^2 for the update."""
    k, n = c["k"], c["n2d"] + c["n3d"] * c["nz"]
    step = c["cube_n"] - c["overlap"]
    cubes = (-(-c["nlat"] // step)) * (-(-c["nlon"] // step))
    cov = (c["cube_n"] / step) ** 2 if c["overlap"] else 1.0
    ncol = c["nlat"] * c["nlon"]
    p = c["n_obs"] * 0.5 * (1.0 - math.cos(min(math.pi, 2.0 * c["dist"] / A_F)))
    chunks = 1
    if c["vert"] > 0:
        chunks = -(-c["nz"] // c["cube_nz"])
        if not c["lnp"]:      # rows beyond the vertical support carry weight 0
            p *= min(1.0, 4.0 * c["vert"] / max(c["nz"] - 1, 1))
    a = cubes * chunks
    fl = a * (k * (k + 1) * p + 2 * k * p + 10.0 / 3.0 * k ** 3 + 4 * k * k)
    fl += 2.0 * k * k * n * ncol * cov
    by = state_bytes * 2.0 * ncol * n * k + 16.0 * ncol * n + c["n_obs"] * (8.0 * k + 48)
    return by, fl


def work(case):
    c = dict(case)
    if c["kind"] == "core":
        k = c["k"]
        rows = c["p"] if c["n"] == 1 else c["p"] * c["n"] / 2.0
        return dict(bytes=rows * (8.0 * k + 20) + c["n"] * 8.0 * (k * k + k),
                    flops=rows * (k * (k + 1.0) + 2 * k) + c["n"] * (10.0 / 3.0 * k ** 3 + 4 * k * k))
    if c["kind"] == "operator":
        rows = c["n_obs"] + c["stations"] * 3.0 * c["nz"]
        n_state = c["nlat"] * c["nlon"] * (1 + 3.0 * c["nz"])
        # no more of the state than the rows touch: 8 points each
        return dict(bytes=min(8.0 * n_state * (c["k"] + 1), 64.0 * rows * (c["k"] + 1))
                    + rows * (8.0 * c["k"] + 40), flops=30.0 * rows * c["k"])
    if c["kind"] == "serve":
        by = fl = 0.0
        for k in (int(s) for s in c["ks"].split(",")):
            cc = _cycle("", nlat=c["nlat"], nlon=c["nlon"], nz=c["nz"], n3d=3, k=k,
                        mix="clustered", n_obs=c["n_obs"], dist=300.0, prec=c["prec"])
            b, f = _cycle_work(cc, 8.0)
            by, fl = by + 3 * b, fl + 3 * f
        return dict(bytes=by, flops=fl)
    by, fl = _cycle_work(c, 8.0 if c["call"] == "run_da" or not c["f32"] else 4.0)
    return dict(bytes=by, flops=fl)


# --------------------------------------------------------------------------
# the same results in 64 bits, in plain torch / numpy
# --------------------------------------------------------------------------

def _gaspari_cohn(r):
    o = torch.zeros_like(r)
    ro = torch.clamp(r, min=0.5)
    rj = (ro / 12.0 - 0.5) * ro + 0.625
    outer = ((rj * ro + C1) * ro - 5.0) * ro + 4.0 - C2 / ro
    inner = (((-0.25 * r + 0.5) * r + 0.625) * r - C1) * r * r + 1.0
    return torch.where(r > 2.0, o, torch.where(r > 1.0, outer, inner))


def _transforms(a, b, rho):
    """T + w 1^T with T = ((k-1) M^-1)^(1/2), w = M^-1 b, M = A + (k-1)/rho I,
    for a batch: LAPACK for a few, else coupled Newton-Schulz iterations."""
    k = a.shape[-1]
    if a.shape[0] * k ** 3 < 2e9:
        lam, v = torch.linalg.eigh(a.cpu())
        lam = lam + (k - 1) / rho
        v, lam = v.to(a.device), lam.to(a.device)
        vt = v.transpose(1, 2).contiguous()
        t = torch.bmm(v * torch.sqrt((k - 1) / lam)[:, None, :], vt)
        w = torch.bmm(v / lam[:, None, :], torch.bmm(vt, b[:, :, None]))
        return t + w
    eye = torch.eye(k, dtype=a.dtype, device=a.device)
    m = a + (k - 1) / rho * eye
    s = m.abs().sum(dim=2).amax(dim=1)[:, None, None]
    y, z = m / s, eye.expand_as(m).contiguous()
    for _ in range(60):
        r = eye - torch.bmm(z, y)
        if float(r.abs().amax()) < 1e-13:
            break
        t = eye + 0.5 * r
        y, z = torch.bmm(y, t), torch.bmm(t, z)
        y, z = 0.5 * (y + y.transpose(1, 2)), 0.5 * (z + z.transpose(1, 2))
    w = torch.bmm(z, torch.bmm(z, b[:, :, None])) / s
    return math.sqrt(k - 1.0) * z / torch.sqrt(s) + w


def _exact_cycle(c, xb, axb, o, glat, glon):
    """xa, axa of one analysis cycle (interior columns; halo columns 0)."""
    dev, k, h, cn = xb.device, c["k"], c["halo"], c["cube_n"]
    nlat, nlon, nz = c["nlat"], c["nlon"], c["nz"]
    step = cn - c["overlap"]
    xa = torch.zeros(xb.shape, dtype=torch.float64, device=dev)
    axa = torch.zeros_like(axb)
    times = torch.zeros(axb.shape[:2], dtype=torch.float64, device=dev)
    rinv = o["rinv"].float().double()
    rows_of = (o["rp"][1:] - o["rp"][:-1]).long()
    sl, so = o["lat"] / 180 * PI_F, o["lon"] / 180 * PI_F
    sc, ss = torch.cos(sl), torch.sin(sl)
    cubes = [(i, min(i + cn, nlon), j, min(j + cn, nlat)) for i in range(0, nlon, step)
             for j in range(0, nlat, step)]
    centre = torch.tensor([[(i + 1 + ei) // 2 - 1, (j + 1 + ej) // 2 - 1] for i, ei, j, ej in cubes],
                          device=dev)
    gla, glo = _t(glat, torch.float64, dev), _t(glon, torch.float64, dev)
    chunks = [(0, nz)]
    if c["vert"] > 0:
        chunks = [(z, min(z + c["cube_nz"], nz)) for z in range(0, nz, c["cube_nz"])]
    n3 = [c["n2d"] + v * nz for v in range(c["n3d"])]
    size = max(1, min(400, int(4e8) // max(1, o["n_sites"])))
    for q0 in range(0, len(cubes), size):
        ctr = centre[q0:q0 + size]
        la, lo = gla[ctr[:, 1]] / 180 * PI_F, glo[ctr[:, 0]] / 180 * PI_F
        v = torch.cos(la)[:, None] * sc[None] * torch.cos(lo[:, None] - so[None]) \
            + torch.sin(la)[:, None] * ss[None]
        gc = _gaspari_cohn(A_F * torch.arccos(torch.clamp(v, max=1.0)) / c["dist"])
        col, site = torch.nonzero(gc > 0, as_tuple=True)
        wgt = gc[col, site]
        del v, gc
        # (column, row) pairs, then padded to the longest list of the group
        rep = rows_of[site]
        col_r, wgt_r = col.repeat_interleave(rep), wgt.repeat_interleave(rep)
        first = o["rp"].long()[site].repeat_interleave(rep)
        at = torch.arange(col_r.numel(), device=dev) - (torch.cumsum(rep, 0) - rep).repeat_interleave(rep)
        row_r = first + at
        n = ctr.shape[0]
        cnt = torch.bincount(col_r, minlength=n)
        pmax = max(1, int(cnt.max()) if cnt.numel() else 1)
        pos = torch.arange(col_r.numel(), device=dev) - (torch.cumsum(cnt, 0) - cnt)[col_r]
        idx = torch.zeros((n, pmax), dtype=torch.int64, device=dev)
        w = torch.zeros((n, pmax), dtype=torch.float64, device=dev)
        idx[col_r, pos] = row_r
        w[col_r, pos] = wgt_r * rinv[row_r]
        sub = max(1, min(n, int(1.5e8) // (pmax * k)))
        for u in range(0, n, sub):
            cub = cubes[q0 + u:q0 + min(u + sub, n)]
            y, ww, id_ = o["yb"][idx[u:u + sub]], w[u:u + sub], idx[u:u + sub]
            yt = y.transpose(1, 2).contiguous()
            for (z0, z1) in chunks:
                wz = ww
                if c["vert"] > 0:
                    mid = (z0 + 1 + z1) // 2
                    if c["lnp"]:
                        hya, hyb = _hybrid(nz)
                        cu = ctr[u:u + sub]
                        ps = axb[cu[:, 0] + h, cu[:, 1] + h, 0]
                        ph = [hya[l] * (P0 - PTOP) + hyb[l] * (ps - PTOP) + PTOP for l in (mid - 1, mid)]
                        zc = torch.log(0.5 * (ph[0] + ph[1]))[:, None]
                    else:
                        zc = float(mid)
                    wz = ww * _gaspari_cohn((zc - o["vco"][id_]).abs() / c["vert"])
                yw = yt * wz[:, None, :]
                a = torch.bmm(yw, y)
                b = torch.bmm(yw, o["dep"][id_][:, :, None])[:, :, 0]
                t = _transforms(0.5 * (a + a.transpose(1, 2)), b, c["rho"])
                el = torch.arange(axb.shape[2], device=dev)
                if c["vert"] > 0:
                    el = [s + l for s in n3 for l in range(z0, z1)]
                    el = torch.tensor((list(range(c["n2d"])) if z1 == nz else []) + el, device=dev)
                if not el.numel():
                    continue
                for di in range(cn):
                    for dj in range(cn):
                        at = [(g, i + di, j + dj) for g, (i, ei, j, ej) in enumerate(cub)
                              if i + di < ei and j + dj < ej]
                        if not at:
                            continue
                        g, ii, jj = torch.tensor(at, device=dev).T
                        ii, jj = ii + h, jj + h
                        f = torch.bmm(xb[ii, jj][:, el].double(), t[g]) + axb[ii, jj][:, el][..., None]
                        m = f.mean(dim=2)
                        xa[ii[:, None], jj[:, None], el[None]] += f - m[..., None]
                        axa[ii[:, None], jj[:, None], el[None]] += m
                        if z0 == 0:
                            times[ii, jj] += 1.0
            del y, yt
    if c["overlap"]:
        times = torch.clamp(times, min=1.0)
        xa, axa = xa / times[..., None, None], axa / times[..., None]
    return xa, axa


def _exact_operator(c, seed):
    xb, axb, o, glat, glon, n = _operator_inputs(c, seed)
    dev, k, nz = xb.device, c["k"], c["nz"]

    def cell(g, close, v):
        edge = torch.cat([_t(g, torch.float64, dev), torch.tensor([close], device=dev).double()])
        t = torch.searchsorted(edge[:-1].contiguous(), v.contiguous())   # 0-based, edge[t] >= v
        lo, hi = edge[torch.clamp(t - 1, min=0)], edge[t]
        d = (hi.float() - lo.float()).double()
        w = torch.where(t == 0, torch.zeros_like(v), (d - v + lo) / torch.where(t == 0, 1.0, d))
        return t, w

    ti, wi = cell(glat, 90.0, o["lat"])
    tj, wj = cell(glon, 360.0, o["lon"])
    x = xb.view(-1, n, k)
    ax = axb.view(-1, n)
    ext = c["nlat"] + 2
    hya, hyb = _hybrid(nz)
    hya, hyb = _t(hya, torch.float64, dev), _t(hyb, torch.float64, dev)
    start = torch.tensor([0, 1, 1 + nz, 1 + 2 * nz], device=dev)
    yb = torch.empty((o["n_rows"], k), dtype=torch.float64, device=dev)
    dep = torch.empty(o["n_rows"], dtype=torch.float64, device=dev)
    for r0 in range(0, o["n_rows"], 20000):
        r = slice(r0, r0 + 20000)
        s, var, ph = o["site"][r], o["var"][r].long(), o["ph"][r]
        ai, aj = wi[s][:, None], wj[s][:, None]
        base = tj[s] * ext + ti[s]                       # the (t - 1, t - 1) point, halo 1

        def bil(el):
            el = el.expand(s.numel(), k)
            e = torch.arange(k, device=dev)[None]
            f = lambda c_: x[c_[:, None], el, e] + ax[c_[:, None], el]  # noqa: E731
            return (f(base) * ai + f(base + 1) * (1 - ai)) * aj \
                + (f(base + ext) * ai + f(base + ext + 1) * (1 - ai)) * (1 - aj)

        zero = torch.zeros((s.numel(), 1), dtype=torch.int64, device=dev)
        ps = bil(zero)
        face = hya * (P0 - PTOP) + hyb * (ps[..., None] - PTOP) + PTOP
        mid = 0.5 * (face[..., :-1] + face[..., 1:])
        pos = (ph[:, None, None] > mid).sum(dim=2)       # levels above the row
        up = torch.clamp(pos, 1, nz - 1)
        lu = torch.log(torch.gather(mid, 2, up[..., None]))[..., 0]
        ll = torch.log(torch.gather(mid, 2, up[..., None] - 1))[..., 0]
        w = (lu - torch.log(ph)[:, None]) / (lu - ll)
        w = torch.where(pos == 0, 1.0, torch.where(pos >= nz, 0.0, w))
        st = start[var][:, None]
        three = (var > 0)[:, None]
        e0 = torch.where(three, st + up - 1, st)
        e1 = torch.where(three, st + up, st)
        val = bil(e0) * w + bil(e1) * (1 - w)
        val = torch.where(three, val, bil(st))
        m = val.mean(dim=1)
        yb[r], dep[r] = val - m[:, None], o["yo"][r] - m
    return [yb, dep]


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "core":
        ts, ws = [], []
        for y, rinv, dep, rloc in _core_inputs(c, seed):
            w = rinv.astype(np.float64) * rloc
            a, b = torch.from_numpy((y * w) @ y.T), torch.from_numpy((y * w) @ dep)
            lam, v = torch.linalg.eigh(0.5 * (a + a.T))
            lam = lam + (c["k"] - 1) / c["rho"]
            wb = v @ ((v.T @ b) / lam)
            ts.append(((v * torch.sqrt((c["k"] - 1) / lam)) @ v.T + wb[:, None]).numpy())
            ws.append(wb.numpy())
        if c["n"] == 1:
            return ts[0], ws[0]
        return np.array(ts), np.array(ws), None
    if c["kind"] == "operator":
        return _exact_operator(c, seed)
    if c["kind"] == "serve":
        out = [None]
        for j in _serve_jobs(c, seed):
            xa, axa = j["xb"], j["axb"]
            for o in j["obs"]:
                xa, axa = _exact_cycle(j["case"], xa, axa, o, j["glat"], j["glon"])
            out.append([xa, axa])
        return out
    xb, axb, o, glat, glon = _cycle_inputs(c, seed)
    if c["call"] != "run_da":
        return [None] + list(_exact_cycle(c, xb, axb, o, glat, glon))
    # the split of the full state, then the polar mask, the blend and the spreads
    x = xb + axb[..., None]
    axb = x.mean(dim=3)
    xb = x - axb[..., None]
    xa, axa = _exact_cycle(c, xb, axb, o, glat, glon)
    h = c["halo"]
    inner = (slice(h, h + c["nlon"]), slice(h, h + c["nlat"]))
    xb, axb, xa, axa = xb[inner], axb[inner], xa[inner], axa[inner]
    polar = (_t(glat, torch.float64, xb.device).abs() > POLAR)[None, :, None, None]
    full = torch.where(polar, xb + axb[..., None],
                       GAMMA1 * (axb[..., None] + xb) + GAMMA2 * (axa[..., None] + xa))
    out = torch.zeros_like(x)
    out[inner] = full
    sb = xb.square().mean(dim=3).sqrt()
    sa = torch.where(polar[..., 0], sb, (full - axa[..., None]).square().mean(dim=3).sqrt())
    return [None, out, sb, sa]
