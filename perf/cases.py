"""What users of this library have it do, as cases that can be timed and checked.

A case is a plain dict.  `prepare` builds what a wave-model program holds before
the call (domains with their grids, the next forcing snapshot, a network), `run`
is one pass through the public entry points (umwm_amd.hip), and `exact` restates
the same pass in 64-bit torch from the model's equations (it shares no code with
the library).  The kinds of case:

  sea        one domain: the next wind snapshot goes in, one dtg is run, and the
             fields an output or coupling step reads come out
  operators  the same dtg through the reference's operator call sequence, ending
             with stress('ocn') as the reference's output step does
  cycle      an assimilation cycle: a spectrum in, one dtg, the spectrum out
  ensemble   many domains of uneven size advanced together (hip.Batch)
  network    a domain served by the learned surrogate
  training   Adam steps of the surrogate on samples of the source kernels

Sizes follow the repository's workloads: the reference's 21x11 namelist grid, the
64x48 regional grid, 720x360 at half a degree, the 2 km hurricane (49 x 72 bins)
and the uneven ensembles (25-49 frequencies, 24-72 directions).
"""
import math

import numpy as np
import torch

from umwm_amd import abi, hip

R_EARTH = 6.371009e6
# what a coupling or output step reads: heights, periods, slopes, momentum
# fluxes and the stresses handed to the atmosphere and ocean
POINT_FIELDS = ("ht", "mwp", "mss", "mwl", "cgmxx", "cgmyy", "ustar", "cd", "taux", "tauy")
OCEAN_FIELDS = ("taux_ocntop", "tauy_ocntop", "epsx_ocn", "epsy_ocn", "epsx_atm", "epsy_atm",
                "taux_snl", "tauy_snl")
MEMBER_FIELDS = ("ht", "mwp", "ustar")


def _case(name, kind, mm, nm, om, pm, precision, dtg, **kw):
    c = dict(name=name, kind=kind, mm=mm, nm=nm, om=om, pm=pm, precision=precision, dtg=dtg,
             dx=1e4, grid="plane", wind="field", land=0.2, depth=3000.0, shelf=True,
             options=False, profile=False, members=0, steps=0)
    c.update(kw)
    if name is None:
        del c["name"]
    return c


def listed():
    return [
        # a coupled limited-area model calling every ten minutes: the reference's own
        # default grid, where launches and latency are all there is
        _case("coupled 21x11 f64", "sea", 21, 11, 37, 36, 8, 600.0, land=0.0, profile=True),
        # the small regional run of the test configurations, an hour
        _case("regional 64x48 f64", "sea", 64, 48, 37, 36, 8, 3600.0, land=0.0, shelf=False,
              depth=4000.0, wind="uniform", profile=True),
        # an ice-covered shelf sea with tides: currents, sea ice and densities as forcing
        _case("shelf sea options f32", "sea", 150, 121, 31, 28, 4, 1800.0, options=True,
              depth=300.0),
        # global half-degree forecast in single precision, ten minutes of it
        _case("global half degree f32", "sea", 720, 360, 37, 36, 4, 600.0, grid="globe",
              land=0.3),
        # global one-degree hindcast in double precision
        _case("global one degree f64", "sea", 360, 180, 37, 36, 8, 1200.0, grid="globe",
              land=0.3),
        # 2 km hurricane with fine spectra: the largest spectra a run carries
        _case("hurricane 2 km f32", "sea", 750, 601, 49, 72, 4, 240.0, dx=2e3, wind="storm",
              land=0.1),
        _case("hurricane 2 km f64", "sea", 450, 361, 49, 72, 8, 240.0, dx=2e3, wind="storm",
              land=0.1),
        # an uneven ensemble in one launch per kernel
        _case("ensemble of 12 f32", "ensemble", 130, 90, 37, 48, 4, 1800.0, members=12,
              wind="uniform"),
        # the reference's call sequence, operator by operator, to its output step
        _case("operators 120x91 f64", "operators", 120, 91, 37, 36, 8, 300.0),
        # restart and assimilation: the spectrum goes in and comes out
        _case("assimilation 64x49 f64", "cycle", 64, 49, 37, 36, 8, 600.0),
        # the surrogate serving a hurricane, and its training
        _case("hurricane with network f32", "network", 420, 341, 49, 72, 4, 240.0, dx=2e3,
              wind="storm", land=0.1),
        _case("network training", "training", 64, 48, 37, 36, 4, 3600.0, land=0.0, shelf=False,
              depth=4000.0, steps=16),
    ]


def _spread(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def draw(rng):
    kind = rng.choice(["sea"] * 6 + ["operators", "cycle", "ensemble", "network", "training"])
    precision = rng.choice([4, 8])
    om, pm = rng.randint(25, 49), 4 * rng.randint(6, 18)
    if kind == "sea":
        points = _spread(rng, 150, 250000 if precision == 4 else 90000)
        shape = _spread(rng, 0.5, 2.0)
        mm, nm = max(12, round(math.sqrt(points * shape))), max(11, round(math.sqrt(points / shape)))
        dx = _spread(rng, 2e3, 3e4)
        if rng.random() < 0.25 and points > 3000:
            return _case(None, kind, mm, nm, om, pm, precision, 600.0, grid="globe",
                         land=rng.uniform(0.1, 0.4))
        return _case(None, kind, mm, nm, om, pm, precision, rng.choice([240.0, 300.0]),
                     dx=round(dx), land=rng.uniform(0.0, 0.35), depth=round(_spread(rng, 40, 5000)),
                     shelf=rng.random() < 0.6, wind=rng.choice(["uniform", "field", "storm"]),
                     options=rng.random() < 0.25, profile=rng.random() < 0.3)
    side = round(_spread(rng, 20, 150))
    if kind == "operators":
        return _case(None, kind, side, side + rng.randint(-5, 9), min(om, 40), min(pm, 48),
                     precision, 300.0)
    if kind == "cycle":
        return _case(None, kind, min(side, 90), min(side, 90) + rng.randint(-5, 9), min(om, 40),
                     min(pm, 48), precision, 300.0)
    if kind == "ensemble":
        return _case(None, kind, side, side + rng.randint(-5, 9), om, pm, precision, 600.0,
                     members=rng.randint(3, 16), wind="uniform")
    if kind == "network":
        return _case(None, kind, 60 + side, 50 + side, om, pm, 4, 240.0, dx=2e3, wind="storm",
                     land=0.1)
    return _case(None, kind, 64, 48, min(om, 40), min(pm, 40), 4, 3600.0, land=0.0, shelf=False,
                 depth=4000.0, steps=rng.randint(4, 16))


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _smooth(rng, xyz, length, waves=24):
    """A smooth zero-mean field of unit spread at positions xyz (..., k)."""
    k = rng.normal(0.0, 1.0 / length, size=(waves, xyz.shape[-1]))
    ph = rng.uniform(0.0, 2 * np.pi, size=waves)
    out = np.zeros(xyz.shape[:-1])
    for a, b in zip(k, ph):
        out += np.cos(xyz @ a + b)
    return out * math.sqrt(2.0 / waves)


class _Inputs:
    """Namelist values, grid and forcing of one domain, arrays (mm, nm)."""


def _inputs(c, seed, member=0):
    # the geography belongs to the case, the weather to the seed: a program runs one
    # grid many times
    rng = np.random.default_rng([int(seed), 977, member])
    place = np.random.default_rng([c["mm"], c["nm"], c["om"], c["pm"], member])
    w = _Inputs()
    mm, nm, om, pm = c["mm"], c["nm"], c["om"], c["pm"]
    if c["kind"] == "ensemble":  # uneven members about the case's size
        mm = max(8, int(mm * place.uniform(0.4, 1.0)))
        nm = max(8, int(nm * place.uniform(0.4, 1.0)))
        om = max(25, om - int(place.integers(0, 12)))
        pm = max(24, pm - 4 * int(place.integers(0, 6)))
    kw = dict(mm=mm, nm=nm, om=om, pm=pm, fmin=0.0313, fmax=2.0, fprog=2.0, dtg=c["dtg"],
              delx=c["dx"], dely=c["dx"], dpt=c["depth"], stokes=1, dmin=10.0,
              wspd0=float(rng.uniform(8.0, 20.0)), wdir0=float(rng.uniform(-3.0, 3.0)))
    w.lon = w.lat = w.z = None
    if c["grid"] == "globe":
        lon = 360.0 / mm * (np.arange(mm) + 0.5)[:, None] * np.ones((1, nm))
        lat = np.ones((mm, 1)) * (-90 + 180.0 / nm * (np.arange(nm) + 0.5))[None, :]
        lo, la = np.radians(lon), np.radians(lat)
        xyz = R_EARTH * np.stack([np.cos(la) * np.cos(lo), np.cos(la) * np.sin(lo), np.sin(la)], -1)
        scale = 1.0e6
        w.lon, w.lat = lon, lat
        kw.update(isglobal=1, gridfromfile=1)
    else:
        x = np.arange(mm)[:, None] * np.ones((1, nm)) * c["dx"]
        y = np.ones((mm, 1)) * np.arange(nm)[None, :] * c["dx"]
        xyz = np.stack([x, y], -1)
        scale = 0.15 * min(mm, nm) * c["dx"]
    if c["land"] > 0 or c["shelf"]:
        depth = np.full((mm, nm), float(c["depth"]))
        if c["shelf"]:  # shallow to deep across the grid, with relief on it
            depth = 10.0 + (depth - 10.0) * (np.arange(mm)[:, None] + 1.0) / mm
            depth *= np.exp(0.3 * _smooth(place, xyz, 0.5 * scale))
        w.z = -np.maximum(depth, 5.0)
        if c["land"] > 0:
            f = _smooth(place, xyz, scale)
            w.z = np.where(f >= np.quantile(f, 1.0 - c["land"]), 1.0, w.z)
        kw.update(topofromfile=1)
    w.storm, w.now, w.next = None, {}, {}
    if c["wind"] != "uniform":
        kw.update(winds=1)
    if c["wind"] == "storm":
        vmax, cx, cy = rng.uniform(45.0, 62.0), 0.5 * mm * c["dx"], 0.55 * nm * c["dx"]
        # a storm moving on with the westerlies: its centre is not becalmed
        tr = (float(rng.uniform(-6, 6)), float(rng.uniform(-16, -12)))
        w.storm = dict(xc=float(cx + tr[0] * c["dtg"]), yc=float(cy + tr[1] * c["dtg"]),
                       vmax=float(vmax), rmax=0.1 * min(mm, nm) * c["dx"], b=1.5, trans=tr)
        u, v = _holland(xyz[..., 0], xyz[..., 1], dict(w.storm, xc=float(cx), yc=float(cy)))
        w.now.update(uw=u, vw=v)
        if c["options"]:  # with more than wind, snapshots are delivered as fields
            u, v = _holland(xyz[..., 0], xyz[..., 1], w.storm)
            w.next.update(uw=u, vw=v)
            w.storm = None
    elif c["wind"] == "field":
        for d, turn in ((w.now, 0.0), (w.next, 0.05)):
            r = np.random.default_rng([int(seed), 31, member])
            speed = kw["wspd0"] * (1 + 0.35 * np.tanh(_smooth(r, xyz, scale)))
            angle = kw["wdir0"] + turn + 0.5 * np.tanh(_smooth(r, xyz, scale))
            d.update(uw=speed * np.cos(angle), vw=speed * np.sin(angle))
    if c["options"]:
        kw.update(currents=1, seaice=1, air_density=1, water_density=1)
        uc, vc = (0.4 * np.tanh(_smooth(rng, xyz, 0.5 * scale)) for _ in range(2))
        ice = np.clip(0.15 + 0.5 * _smooth(rng, xyz, scale), 0.0, 1.0)
        ra = 1.2 * (1 + 0.04 * np.tanh(_smooth(rng, xyz, scale)))
        rw = 1025.0 * (1 + 0.004 * np.tanh(_smooth(rng, xyz, scale)))
        for d, f in ((w.now, 1.0), (w.next, 0.9)):
            d.update(uc=f * uc, vc=f * vc, fice=f * ice, rhoa=ra, rhow=rw)
    w.c, w.kw = c, kw
    w.forced = any(kw.get(k) for k in ("winds", "currents", "seaice"))
    w.alpha = float(rng.uniform(0.006, 0.014))
    return w


def _holland(x, y, s):
    """Holland (1980) wind as umwm_hip_holland_forcinginput defines it."""
    rho, f = 1.15, 2 * 7.292e-5 * math.sin(math.radians(20.0))
    dp = rho * math.e * s["vmax"] ** 2 / s["b"]
    r = np.hypot(x - s["xc"], y - s["yc"]) + 1.0
    a = (s["rmax"] / r) ** s["b"]
    v = np.sqrt(s["b"] * dp / rho * a * np.exp(-a) + (r * f / 2) ** 2) - r * f / 2
    th = np.arctan2(y - s["yc"], x - s["xc"]) + np.pi / 2 + math.radians(20.0)
    return v * np.cos(th) + 0.5 * s["trans"][0], v * np.sin(th) + 0.5 * s["trans"][1]


def _weights(c, seed):
    """A network of the library's shape, as loaded from a file."""
    g = np.random.default_rng([int(seed), 5])
    nb = c["om"] * c["pm"]
    dims = [nb + 3, 512, 512, 512, nb]
    out = []
    for l in range(4):
        # a network in use departs little from the mean of each output
        gain = 0.05 if l == 3 and c["kind"] == "network" else 1.0
        w = g.standard_normal((dims[l + 1], dims[l]), dtype=np.float32)
        w *= np.float32(gain / math.sqrt(dims[l]))
        out.append((w, np.zeros(dims[l + 1], np.float32)))
    return out


# ---------------------------------------------------------------------------
# the passes
# ---------------------------------------------------------------------------
def _domain(w):
    grid = abi.make_grid_input(lon=w.lon, lat=w.lat, z=w.z)
    forcing = abi.make_forcing_input(**w.now) if w.forced else None
    d = hip.Domain(abi.make_params(**w.kw), grid, forcing, precision=w.c["precision"])
    d.init_jonswap(abi.make_jonswap(alpha=w.alpha, fp_from_wind=True))
    d.stokes_drift(True)
    if w.c["kind"] == "operators":
        d.operator_substep()
    else:
        d.substep()  # the cold first substep (dts = 0)
    return d


class _State:
    def __del__(self):
        for name in ("batch", "net"):
            if getattr(self, name, None) is not None:
                getattr(self, name).close()
        for d in getattr(self, "domains", ()):
            d.close()


def prepare(case, seed):
    s = _State()
    s.case = case
    s.inputs = [_inputs(case, seed, k) for k in range(max(1, case["members"]))]
    s.domains = [_domain(w) for w in s.inputs]
    w, d = s.inputs[0], s.domains[0]
    s.storm = abi.make_holland(**w.storm) if w.storm else None
    s.next = abi.make_forcing_input(**w.next) if w.forced and not w.storm else None
    if case["kind"] == "ensemble":
        s.batch = hip.Batch(s.domains)
    if case["kind"] == "cycle":
        rng = np.random.default_rng([int(seed), 3])
        s.analysis = d.get("e") * rng.uniform(0.9, 1.1, size=(d.im, 1, 1))
        s.ustar = d.get("ustar")
    if case["kind"] in ("network", "training"):
        if case["kind"] == "network":
            d.run_dtg()  # the sea has left its initial spectrum when samples are taken
        s.net = hip.Surrogate(abi.make_surrogate_config(
            om=case["om"], pm=case["pm"], batch=2048, chunk=65536 if case["kind"] == "network" else 2048,
            capacity=d.im, seed=int(seed) % 1000 + 1))
        s.net.collect(d)
        if case["kind"] == "network":
            s.net.train(1, lr=1e-6)  # fixes the normalisation of the inputs and outputs
        for l, (a, b) in enumerate(_weights(case, seed)):
            s.net.set_layer(l, a, b)
        if case["kind"] == "network":
            # a policy that lets the network serve every point
            s.net.attach(d, abi.make_surrogate_policy(resid_tol=10.0, audit_tol=1e6,
                                                      range_margin=1e3, zmax=1e6))
    return s


def _read(case, d, names):
    """Fields as a program keeps them: in the domain's precision."""
    t = np.float32 if case["precision"] == 4 else np.float64
    return {n: np.asarray(d.get(n), dtype=t) for n in names}


def run(state):
    c, d = state.case, state.domains[0]
    if c["kind"] == "training":
        state.net.train(c["steps"], lr=1e-4)
        # the bfloat16 copies that the network multiplies with
        return {"layer%d" % l: [torch.from_numpy(a).bfloat16() for a in state.net.get_layer(l)]
                for l in range(state.net.layers + 1)}
    if c["kind"] == "ensemble":
        state.batch.run_dtg()
        return [_read(c, m, MEMBER_FIELDS) for m in state.domains]
    if state.storm is not None:
        d.holland_forcinginput(state.storm)
    elif state.next is not None:
        d.forcinginput(state.next)
    if c["kind"] == "operators":
        d.set_scalar("sumt", 0.0)
        while d.scalar("sumt") < c["dtg"]:
            d.operator_substep()
        d.stress("ocn")
        d.stokes_drift()
        d.diag()
        return _read(c, d, POINT_FIELDS + OCEAN_FIELDS)
    if c["kind"] == "cycle":
        d.set("e", state.analysis)
        d.set("ustar", state.ustar)
        d.run_dtg()
        return _read(c, d, ("e", "ustar", "ht"))
    d.run_dtg()
    return _read(c, d, POINT_FIELDS + (("us", "vs") if c["profile"] else ()))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    c = case
    nb, size = c["om"] * c["pm"], c["precision"]
    points = c["mm"] * c["nm"] * (1.0 - c["land"])
    if c["kind"] == "training":
        params = (nb + 3) * 512 + 2 * 512 * 512 + 512 * nb
        return {"bytes": c["steps"] * (2048.0 * (2 * nb + 3) * 4 + params * 28.0),
                "flops": c["steps"] * 2048.0 * 6.0 * params}
    if c["kind"] == "ensemble":
        points *= 0.49 * c["members"]
        nb *= 0.72
    # substeps: the advective limit of the longest wave (or of the polar rows), and
    # about 80 s where the source terms limit the step
    cg = min(math.sqrt(9.81 * c["depth"]), 25.0)
    dx = c["dx"] if c["grid"] == "plane" else 2 * math.pi * R_EARTH / c["mm"] * math.cos(
        math.pi / 2 * (1 - 3.0 / c["nm"]))
    n = max(1.0, math.ceil(c["dtg"] / min(80.0, 0.7 * dx / cg)))
    bins = points * nb
    # per substep every bin is read once and written once; some 70 operations and three
    # transcendentals of about 20 make a bin's new value
    out = {"bytes": n * 2.0 * bins * size, "flops": n * bins * 130.0}
    if c["kind"] == "network":
        params = (nb + 3) * 512 + 2 * 512 * 512 + 512 * nb
        out["flops"] += n * points * 2.0 * params
    if c["kind"] == "cycle":
        out["bytes"] += 4.0 * bins * 8
    return out


# ---------------------------------------------------------------------------
# the same passes in 64 bits: the model's equations in plain torch
# ---------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _tensor(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_dev())


class _Sea:
    """One domain's equations in float64, sea points in column order with one
    land point appended (index n) that neighbours on land refer to."""

    def __init__(self, w):
        self.p = p = dict(abi.DEFAULTS, **w.kw)
        self.w = w
        mm, nm, om, pm = p["mm"], p["nm"], p["om"], p["pm"]
        mask = np.ones((mm, nm), bool)
        mask[:, [0, -1]] = False
        if not p["isglobal"]:
            mask[[0, -1], :] = False
        d2 = np.full((mm, nm), float(p["dpt"]))
        if p["topofromfile"]:
            d2 = np.maximum(np.abs(w.z), p["dmin"])
            mask &= w.z < 0
        self.mask = mask
        dx2, dy2, curv = np.full((mm, nm), float(p["delx"])), np.full((mm, nm), float(p["dely"])), np.zeros((mm, nm))
        if p["gridfromfile"]:
            dx2, dy2, curv = self._metric(np.radians(w.lon), np.radians(w.lat))
        m, n = np.nonzero(mask)
        self.n = im = len(m)
        index = np.full((mm, nm), im)
        index[m, n] = np.arange(im)
        east, west = (m + 1) % mm, (m - 1) % mm
        near = ((east, n), (west, n), (m, n + 1), (m, n - 1))
        self.ie, self.iw, self.iN, self.iS = (torch.as_tensor(index[q], device=_dev()) for q in near)
        T = _tensor
        self.near_cells, self.cell = near, (m, n)
        self.dx, self.dy, self.d = T(dx2[m, n]), T(dy2[m, n]), T(d2[m, n])
        self.dye, self.dyw = (0.5 * (self.dy + T(dy2[q])) for q in near[:2])
        self.dxn, self.dxs = (0.5 * (self.dx + T(dx2[q])) for q in near[2:])
        self.curv = T(curv[m, n])
        dlnf = (math.log(p["fmax"]) - math.log(p["fmin"])) / (om - 1)
        self.f = [math.exp(math.log(p["fmin"]) + o * dlnf) for o in range(om)]
        self.dlnf, self.dth = dlnf, 2 * math.pi / pm
        self.th = T([(q + 1 - 0.5 * (pm + 1)) * self.dth for q in range(pm)])[:, None]
        self.ct, self.st = torch.cos(self.th), torch.sin(self.th)
        b1, b2 = math.exp(-16 * dlnf ** 2), math.exp(-64 * dlnf ** 2)
        self.bf1, self.bf2 = b1 / (b1 + b2), b2 / (b1 + b2)
        self._dispersion()
        cfl = math.cos(0.25 * math.pi - 0.5 * self.dth) if pm % 8 == 0 else 1 / math.sqrt(2.0)
        self.dtamin = 0.98 * cfl * min(dx2[mask].min(), dy2[mask].min()) / float(self.cg.max())
        zero = torch.zeros(im, dtype=torch.float64, device=_dev())
        self.us1, self.vs1 = zero, zero
        self.now = self.next = w.now
        if p["winds"]:
            self.wspd, self.wdir = T(np.hypot(w.now["uw"], w.now["vw"])[m, n]), zero
        else:
            self.wspd, self.wdir = zero + p["wspd0"], zero + p["wdir0"]
        self.uc, self.vc = zero + p["uc0"], zero + p["vc0"]
        self.rhoa, self.rhow = zero + p["rhoa0"], zero + p["rhow0"]
        self.fice = zero + p["fice0"]
        self.dv = self.du = zero
        cd = torch.where(self.wspd > 11, (0.49 + 0.065 * self.wspd) * 1e-3, zero + 1.2e-3)
        self.ustar = torch.sqrt(cd) * self.wspd
        self._jonswap(w.alpha)
        self.dm_net = None
        self.first = True

    @staticmethod
    def _metric(lon, lat):
        def dist(lo1, lo2, la1, la2):
            s1, s2 = np.sin(0.5 * np.abs(la2 - la1)), np.sin(0.5 * np.abs(lo2 - lo1))
            return 2 * R_EARTH * np.arcsin(np.sqrt(s1 ** 2 + np.cos(la1) * np.cos(la2) * s2 ** 2))

        dx, dy = np.zeros_like(lon), np.zeros_like(lon)
        lo, la = 0.5 * (lon[1:] + lon[:-1]), 0.5 * (lat[1:] + lat[:-1])
        dx[1:-1] = dist(lo[:-1], lo[1:], la[:-1], la[1:])
        dx[0], dx[-1] = 2 * dx[1] - dx[2], 2 * dx[-2] - dx[-3]
        lo, la = 0.5 * (lon[:, 1:] + lon[:, :-1]), 0.5 * (lat[:, 1:] + lat[:, :-1])
        dy[:, 1:-1] = dist(lo[:, :-1], lo[:, 1:], la[:, :-1], la[:, 1:])
        dy[:, 0], dy[:, -1] = 2 * dy[:, 1] - dy[:, 2], 2 * dy[:, -2] - dy[:, -3]
        lw, le = np.roll(lon, 1, 0), np.roll(lon, -1, 0)
        aw, ae = np.roll(lat, 1, 0), np.roll(lat, -1, 0)
        turn = np.arctan2(np.sin(le - lw) * np.cos(ae),
                          np.cos(aw) * np.sin(ae) - np.sin(aw) * np.cos(ae) * np.cos(le - lw))
        return dx, dy, turn - 0.5 * np.pi

    def _dispersion(self):
        p, d, g = self.p, self.d, self.p["g"]
        f = _tensor(self.f)[:, None]
        b = p["sfct"] / (p["rhow0"] * g * d ** 2)
        fn = 2 * math.pi * torch.sqrt(d / g) * f
        kk = fn ** 2
        go = torch.ones_like(kk, dtype=torch.bool)
        while go.any():  # Newton steps until one is at most 0.01
            t = torch.tanh(kk)
            dk = -(fn ** 2 - kk * t * (1 + b * kk ** 2)) / (
                3 * b * kk ** 2 * t + t + kk * (1 + b * kk ** 2) * (1 - t ** 2))
            kk = torch.where(go, kk - dk, kk)
            go = go & (dk.abs() > 1e-2)
        self.k = k = kk.abs() / d
        kd = torch.clamp(k * d, max=20.0)
        sk2 = p["sfct"] * k ** 2
        cp = 2 * math.pi * f / k
        cg = cp * (0.5 + k * d / torch.sinh(2 * kd) + sk2 / (p["rhow0"] * g + sk2))
        self.dwn = 2 * math.pi * self.dlnf * f / cg.abs()
        self.kdk = k * self.dwn
        self.coth = 1 / torch.tanh(0.2 * kd)
        self.sbf = p["sbf_fac"] * k / torch.sinh(2 * kd) + p["sbp_fac"] * k / torch.cosh(kd) ** 2
        self.logl = torch.log(torch.clamp(0.5 * cp / f, max=20.0) / p["z"])
        ghost = lambda a: torch.cat([a, a.min(1, keepdim=True).values], 1)  # noqa: E731
        self.cp, self.cg = ghost(cp), ghost(cg)

    def _jonswap(self, alpha):
        p, g = self.p, self.p["g"]
        fp = torch.clamp(0.13 * g / torch.clamp(self.wspd, min=3.0), 0.05, 0.5)
        c = torch.cos(self.th - self.wdir)
        spread = torch.where(c > 0, 2 / math.pi * c * c, torch.zeros_like(c))
        self.e = torch.empty(p["om"], p["pm"], self.n, dtype=torch.float64, device=_dev())
        for o, fo in enumerate(self.f):
            sig = torch.where(fp >= fo, torch.full_like(fp, 0.07), torch.full_like(fp, 0.09))
            r = torch.exp(-(fo - fp) ** 2 / (2 * sig ** 2 * fp ** 2))
            s = alpha * g * g * (2 * math.pi) ** -4 * fo ** -5 * torch.exp(-1.25 * (fp / fo) ** 4) * 3.3 ** r
            self.e[o] = s * fo * self.dlnf * spread / self.kdk[o]

    def level(self, snapshot):
        self.now, self.next = self.next, snapshot

    def _forcing(self, s):
        p, x = self.p, s / self.p["dtg"]

        def at(name, cells, sea_only=False):
            v = _tensor((1 - x) * self.now[name][cells] + x * self.next[name][cells])
            return v * _tensor(self.mask[cells]) if sea_only else v

        if p["winds"]:
            u, v = at("uw", self.cell), at("vw", self.cell)
            self.wspd, self.wdir = torch.sqrt(u * u + v * v), torch.atan2(v, u)
        if p["currents"]:
            self.uc, self.vc = at("uc", self.cell, True), at("vc", self.cell, True)
            self.ncur = [(at("uc", q, True), at("vc", q, True)) for q in self.near_cells]
        if p["seaice"]:
            self.fice = at("fice", self.cell)
        if p["air_density"]:
            self.rhoa = at("rhoa", self.cell)
        if p["water_density"]:
            self.rhow = at("rhow", self.cell)

    def _near(self, a, index):
        """Values at neighbours of sea-point rows a (..., n); land holds none."""
        return torch.cat([a, torch.zeros_like(a[..., :1])], -1)[..., index]

    def _moment_steps(self):
        """Per frequency, the directional convolution of all lower ones."""
        z = torch.zeros(self.n, dtype=torch.float64, device=_dev())
        m0, mc, ms = z, z, z
        c2, s2 = self.ct ** 2 - self.st ** 2, 2 * self.ct * self.st
        for o in range(self.p["om"]):
            yield o, 0.5 * self.dth * (m0 + c2 * mc + s2 * ms), 0.5 * self.dth * m0
            k3 = self.k[o] ** 2 * self.kdk[o]
            m0 = m0 + k3 * self.e[o].sum(0)
            mc = mc + k3 * (c2 * self.e[o]).sum(0)
            ms = ms + k3 * (s2 * self.e[o]).sum(0)

    def _source_input(self, o, oc):
        p = self.p
        cw = torch.cos(self.wdir - self.th)
        x = (self.wspd + 2.5 * self.ustar * self.logl[o]) * cw - self.cp[o, :-1] - self.uc * self.ct - self.vc * self.st
        y = x.abs() * x
        one = torch.ones_like(cw)
        against = torch.where(cw > 0, p["sin_diss2"] * one, p["sin_diss1"] * one)
        y = y * torch.where(y > 0, self.shelt.expand_as(y), against)
        s = (1 - self.fice) * 2 * math.pi * self.rhoa / self.rhow * y * self.f[o] * self.k[o] / p["g"]
        return torch.where(oc < o, torch.clamp(s, min=0.0), s)

    def _spreading(self, o, mss, m0):
        p = self.p
        dm = (1 + p["mss_fac"] * mss) ** 2
        if self.dm_net is not None:
            hi = (1 + 2 * p["mss_fac"] * m0) ** 2
            net = 1 + self.dm_net[:, o * p["pm"]:(o + 1) * p["pm"]].T
            dm = torch.minimum(torch.clamp(net, min=1.0), hi.expand_as(net))
        return dm

    def substep(self, sumt):
        p, om, n = self.p, self.p["om"], self.n
        if self.w.forced:
            self._forcing(sumt)
        if self.net is not None:
            self.dm_net = self.net(self)
        self.wspd = torch.clamp(self.wspd, min=1e-2)
        self.shelt = _sheltering(self.wspd)
        fc = torch.clamp(0.53 * p["g"] / self.wspd, max=p["fprog"])
        oc = torch.zeros(n, dtype=torch.int64, device=_dev())
        for o in range(om - 2):
            oc = torch.where(fc > self.f[o], o, oc)
        root = torch.sqrt(self.rhoa / self.rhow)
        hs = 4 * torch.sqrt((self.e.sum(1) * self.kdk).sum(0) * self.dth)
        ice = torch.where(self.fice > p["fice_lth"], -5.35e-6 * torch.clamp(hs, max=3.0), 0.0)
        tp, pw = 2 * math.pi * p["sds_fac"], p["sds_power"]
        B1 = p["snl_fac"] * self.bf1 * self.kdk[1:-1] / self.kdk[:-2]
        B2 = p["snl_fac"] * self.bf2 * self.kdk[2:] / self.kdk[:-2]

        def losses(o):
            tail = p["sdt_fac"] * root * self.ustar * self.k[o] + 4 * p["nu_water"] * self.k[o] ** 2 - 2 * self.cg[o, :-1] * ice
            return self.sbf[o] + tail, tail

        # the step: the largest rate of any prognostic bin
        most = torch.zeros(n, dtype=torch.float64, device=_dev())
        for o, mss, m0 in self._moment_steps():
            sds = tp * self.f[o] * self._spreading(o, mss, m0) * (self.e[o].abs() * self.k[o] ** 4) ** pw * self.coth[o]
            share = 1 - (B1[o] + B2[o]) if o < om - 2 else 0.0
            r = self._source_input(o, oc) - sds * share - losses(o)[0]
            most = torch.maximum(most, torch.where(oc >= o, r.abs().max(0).values, 0.0))
        dts = min(float((p["explim"] / most).min()), self.dtamin, p["dtg"] - sumt)
        if self.first:
            dts = 0.0
        if p["currents"] or self.first:
            self._rotation(oc, dts)
        # integration, with the downshift of each bin into the two below it
        half = torch.empty_like(self.e)  # (E^n + E_s) / 2
        X, full = [], []
        for o, mss, m0 in self._moment_steps():
            dm = self._spreading(o, mss, m0)
            s = tp * self.f[o] * dm * (self.e[o].abs() * self.k[o] ** 4) ** pw
            X.append(s * self.e[o])
            ss = self._source_input(o, oc)
            crest, tail = losses(o)
            grown = self.e[o] * torch.exp(dts * (ss - s * self.coth[o] - crest)) - dts * p["snl_fac"] * X[o]
            t = torch.clamp(ss - tail, min=0.0) / (tp * self.f[o] * dm * self.coth[o])
            full.append(torch.where(oc >= o, grown, t ** (1 / pw) / self.k[o] ** 4))
            for back, B in ((1, B1), (2, B2)):
                q = o - back
                if q >= 0 and q < om - 2:
                    full[q] = full[q] + torch.where(oc >= q, dts * B[q] * X[o], 0.0)
            if o >= 2:
                half[o - 2] = 0.5 * (self.e[o - 2] + full[o - 2])
                X[o - 2] = full[o - 2] = None
        for o in (om - 2, om - 1):
            half[o] = 0.5 * (self.e[o] + full[o])
        self._advance(half, oc, dts)
        self._stress_atm(oc)
        self.oc = oc
        self.first = False
        return dts

    def _rotation(self, oc, dts):
        self.oc_rot = oc
        self.dv = self.du = torch.zeros_like(self.d)
        if self.p["currents"]:
            (_, ve), (_, vw), (un, _), (us, _) = self.ncur
            self.dv, self.du = ve - vw, un - us
        most = 0.0  # bins above the cut-off hold 0 and join the maximum
        for o in range(self.p["om"]):
            r = torch.where(oc >= o, self._rate(o), 0.0)
            most = max(most, float(r.max()))
        self.dtr_most = dts if most <= 2.2250738585072014e-308 else self.dth / most

    def _rate(self, o):
        cp = self.cp[o]
        return 0.5 * (((cp[self.ie] - cp[self.iw]) * self.st + self.dv) / self.dx
                      - ((cp[self.iN] - cp[self.iS]) * self.ct + self.du) / self.dy)

    def _advance(self, half, oc, dts):
        p = self.p
        cc, sc = torch.cos(self.th + self.curv), torch.sin(self.th + self.curv)
        dtr = min(self.dtr_most, dts)
        up = lambda v: (v + v.abs(), v - v.abs())  # noqa: E731
        edges = ((self.ie, self.dye, cc, 1), (self.iw, self.dyw, cc, -1),
                 (self.iN, self.dxn, sc, 1), (self.iS, self.dxs, sc, -1))
        for o in range(p["om"]):
            E, cg = half[o], self.cg[o]
            flux = torch.zeros_like(E)
            for q, (index, width, turn, sign) in enumerate(edges):
                En = self._near(E, index)
                speeds = [(cg[:-1] + cg[index]) * turn]
                if p["currents"]:
                    speeds.append(self.uc + self.ncur[q][0] if q < 2 else self.vc + self.ncur[q][1])
                for v in speeds:
                    a, b = up(v)
                    flux += sign * width * (a * (E if sign > 0 else En) + b * (En if sign > 0 else E))
            rate = torch.where(self.oc_rot >= o, self._rate(o), 0.0)
            rl, rr = 0.5 * (rate + rate.roll(-1, 0)), 0.5 * (rate + rate.roll(1, 0))
            a, b = up(rl)
            c, d = up(rr)
            turn = 0.5 * (a * E + b * E.roll(-1, 0) - c * E.roll(1, 0) - d * E) / self.dth
            new = 2 * E - self.e[o]
            moved = new - 0.25 * dts * flux / (self.dx * self.dy) - dtr * turn
            moved = torch.where(self.fice > p["fice_uth"], torch.zeros_like(moved), moved)
            self.e[o] = torch.where(oc >= o, moved, new)

    def _stress_atm(self, oc):
        p = self.p
        z = torch.zeros_like(self.d)
        sx, sy = z, z
        for o in range(p["om"]):
            v = self.e[o] * self._source_input(o, oc)
            before = torch.cat([self.cp[o, -1:], self.cp[o, :-2]])  # the point one earlier
            tx, ty = (v * self.ct).sum(0) / before, (v * self.st).sum(0) / before
            sx, sy = sx + tx * self.kdk[o], sy + ty * self.kdk[o]
        w, kom, unit = self.wspd, self.k[-1], self.rhow * self.dth * p["g"]
        tail = _tail(w, kom)
        fx, fy = (sx + tx * kom * tail) * unit, (sy + ty * kom * tail) * unit
        u, v = w * torch.cos(self.wdir) - self.uc - self.us1, w * torch.sin(self.wdir) - self.vc - self.vs1
        wr = torch.sqrt(u * u + v * v)
        z0 = torch.full_like(w, 1e-3)
        for _ in range(6):
            us = p["kappa"] * wr / torch.log(p["z"] / z0)
            z0 = 0.132 * p["nu_air"] / us
        form = torch.sqrt(fx * fx + fy * fy) / (self.rhoa * w * w)
        skin = us * us / (w * w)
        skin = torch.clamp(skin * (1 + 2 * skin / (skin + form + 2.3e-308)) / 3, max=1e-2)
        ang = torch.atan2(v, u)
        self.skin = tuple(self.rhoa * skin * wr * wr * t for t in (torch.cos(ang), torch.sin(ang)))
        self.taux, self.tauy = fx + self.skin[0], fy + self.skin[1]
        total = torch.sqrt(self.taux ** 2 + self.tauy ** 2)
        self.cd, self.ustar = total / (self.rhoa * w * w), torch.sqrt(total / self.rhoa)

    net = None

    def run_dtg(self):
        s = 0.0
        while s < self.p["dtg"]:
            s += self.substep(s)

    def stokes(self):
        us, vs = [], []
        a, b = (self.e * self.ct).sum(1), (self.e * self.st).sum(1)
        f, d, k = _tensor(self.f)[:, None] * 2 * math.pi, self.d, self.k
        for depth in abi.DEFAULT_DEPTHS:
            z = -depth
            kd = k * d
            arg = 2 * k * (z + d)
            deep = (arg.abs() > 50) | (kd > 50)
            t = torch.where(deep, 2 * torch.exp(2 * k * z),
                            torch.cosh(torch.clamp(arg, max=50.0)) / torch.sinh(torch.clamp(kd, max=50.0)) ** 2)
            t = torch.where(d >= depth, f * k ** 2 * t * self.dwn * self.dth, torch.zeros_like(t))
            us.append((t * a).sum(0))
            vs.append((t * b).sum(0))
        self.us, self.vs = torch.stack(us), torch.stack(vs)
        self.us1, self.vs1 = us[0], vs[0]

    def diag(self):
        f, g = _tensor(self.f)[:, None], self.p["g"]
        s = self.e.sum(1) * self.kdk
        m0, m2, mk = s.sum(0), (f ** 2 * s).sum(0), (s * self.k ** 2).sum(0)
        self.ht, self.mwp = 4 * torch.sqrt(m0 * self.dth), torch.sqrt(m0 / m2)
        self.mss, self.mwl = mk * self.dth, 2 * math.pi * torch.sqrt(m0 / mk)
        o = torch.arange(self.p["om"], device=_dev())[:, None]
        low = torch.where(self.oc >= o, self.kdk * self.cg[:, :-1] / self.cp[:, :-1], 0.0)
        self.cgmxx, self.cgmyy = (((self.e * t ** 2).sum(1) * low).sum(0) * self.rhow * self.dth * g
                                  for t in (self.ct, self.st))

    def ocean(self, sources):
        """stress('ocn') from the source terms of the last evaluation."""
        p, icp = self.p, 1 / self.cp[:, :-1]
        ustar0, ssin, sds, snl = sources
        z = torch.zeros_like(self.d)
        v = {n: [z, z] for n in ("top", "snl", "epso", "epsa")}
        root = torch.sqrt(self.rhoa / self.rhow)
        for o in range(p["om"]):
            more = p["sdt_fac"] * root * ustar0 * self.k[o] + 4 * p["nu_water"] * self.k[o] ** 2
            lost, heat = self.e[o] * (sds[o] + more), self.e[o] * sds[o]
            if o >= 2:
                cp = self.cp[o, :-1]
                keep = self.bf1 * cp * icp[o - 1] + self.bf2 * cp * icp[o - 2]
                gone = self.bf1 * (1 - cp * icp[o - 1]) + self.bf2 * (1 - cp * icp[o - 2])
                lost, heat = lost - snl[o] * keep, heat - snl[o] * keep
            for i, t in enumerate((self.ct, self.st)):
                last = (lost * t).sum(0) * icp[o]
                v["top"][i] = v["top"][i] + last * self.kdk[o]
                v["epso"][i] = v["epso"][i] + (heat * t).sum(0) * self.kdk[o]
                v["epsa"][i] = v["epsa"][i] + (self.e[o] * ssin[o] * t).sum(0) * self.kdk[o]
                if o >= 2:
                    v["snl"][i] = v["snl"][i] + torch.where(
                        self.oc >= o, (snl[o] * gone * t).sum(0) * icp[o] * self.kdk[o], 0.0)
                if o == p["om"] - 1:
                    v["top"][i] = v["top"][i] + last * self.k[o] * _tail(self.wspd, self.k[o])
        unit = self.rhow * self.dth * p["g"]
        for i, x in enumerate("xy"):
            setattr(self, "tau%s_ocntop" % x, v["top"][i] * unit + self.skin[i])
            setattr(self, "eps%s_ocn" % x, v["epso"][i] * unit)
            setattr(self, "eps%s_atm" % x, v["epsa"][i] * unit)
            setattr(self, "tau%s_snl" % x, v["snl"][i] * unit)

    def sources(self, oc):
        p, om = self.p, self.p["om"]
        tp = 2 * math.pi * p["sds_fac"]
        ssin, raw = [], []
        for o, mss, m0 in self._moment_steps():
            ssin.append(self._source_input(o, oc))
            raw.append(tp * self.f[o] * self._spreading(o, mss, m0) * (self.e[o].abs() * self.k[o] ** 4) ** p["sds_power"])
        snl = []
        for o in range(om):
            v = torch.zeros_like(self.e[o])
            if o < om - 2:
                s = p["snl_fac"] / self.kdk[o]
                v = (s * self.bf1 * self.kdk[o + 1] * raw[o + 1] * self.e[o + 1]
                     + s * self.bf2 * self.kdk[o + 2] * raw[o + 2] * self.e[o + 2]
                     - p["snl_fac"] * raw[o] * self.e[o])
            snl.append(torch.where(oc >= o, v, 0.0))
        return self.ustar, ssin, [r * self.coth[o] for o, r in enumerate(raw)], snl


def _sheltering(w):
    s1, s2 = (0.10 - 0.04) / 15, (0.06 - 0.09) / 27
    c = 0.65 * (s2 - s1) / 18
    b = s1 - 2 * c * 15
    a = 0.10 - b * 15 - c * 225
    last = a + b * 33 + c * 33 ** 2
    return torch.where(w <= 15, 0.04 + s1 * w, torch.where(
        w <= 33, a + b * w + c * w * w, last * torch.exp(-(w - 33) / (1.6 * w))))


def _tail(w, k):
    t = 0.000112 * w * w - 0.01451 * w - 1.0186
    return (1e3 ** (t + 1) - k * k ** t) / (k ** t * (t + 1))


def _gelu(z):
    return 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))


class _Samples:
    """Inputs, targets and their normalisation, of a sea's current state."""

    def __init__(self, sea):
        self.x = self.features(sea)
        t = [((1 + sea.p["mss_fac"] * mss) ** 2).log() for _, mss, _ in sea._moment_steps()]
        self.t = torch.cat(t).T

        def spread(a, floor):
            s = a.std(0, unbiased=False)
            return torch.where(s == 0, 1.0, s).clamp(min=floor)

        self.mu, self.sd = self.x.mean(0), spread(self.x, 0.1)
        self.tmu, self.tsd = self.t.mean(0), spread(self.t, 0.005)

    @staticmethod
    def features(sea):
        w = torch.clamp(sea.wspd, min=1e-2)
        e = torch.log(torch.clamp(sea.e.reshape(-1, sea.n), min=1e-30))
        u, v = w * torch.cos(sea.wdir), w * torch.sin(sea.wdir)
        return torch.cat([e, torch.stack([u, v, torch.log(sea.d)])]).T


def _exact_training(c, seed, sea):
    data = _Samples(sea)
    X, Y = (data.x - data.mu) / data.sd, (data.t - data.tmu) / data.tsd
    W = [_tensor(a).requires_grad_() for layer in _weights(c, seed) for a in layer]
    M, V = [torch.zeros_like(a) for a in W], [torch.zeros_like(a) for a in W]
    r = np.arange(2048, dtype=np.uint64)
    with np.errstate(over="ignore"):
        for k in range(c["steps"]):  # rows are drawn by a hash of seed, step and row
            h = np.uint64(int(seed) % 1000 + 1) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(k) * np.uint64(0xD1B54A32D192ED03)
            x = (h ^ (r * np.uint64(0x632BE59BD9B4E019))) + np.uint64(0x9E3779B97F4A7C15)
            x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            rows = torch.as_tensor(((x ^ (x >> np.uint64(31))) % np.uint64(sea.n)).astype(np.int64), device=_dev())
            a = X[rows]
            for l in range(4):
                a = a @ W[2 * l].T + W[2 * l + 1]
                a = _gelu(a) if l < 3 else a
            grads = torch.autograd.grad(((a - Y[rows]) ** 2).mean(), W)
            with torch.no_grad():
                for a, g, m, v in zip(W, grads, M, V):
                    m.mul_(0.9).add_(0.1 * g)
                    v.mul_(0.999).add_(0.001 * g * g)
                    a -= 1e-4 * m / (1 - 0.9 ** (k + 1)) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    W = [a.detach() for a in W]
    return {"layer%d" % l: [W[2 * l], W[2 * l + 1]] for l in range(4)}


def exact(case, seed):
    c = case
    outs = []
    for member in range(max(1, c["members"])):
        w = _inputs(c, seed, member)
        sea = _Sea(w)
        sea.stokes()
        sea.substep(0.0)
        if c["kind"] == "training":
            return _exact_training(c, seed, sea)
        if c["kind"] == "network":
            sea.run_dtg()
            sea.stokes()
            data = _Samples(sea)
            W = [_tensor(a) for layer in _weights(c, seed) for a in layer]

            def net(sea):
                out = []
                for x in _Samples.features(sea).split(16384):
                    a = (x - data.mu) / data.sd
                    for l in range(4):
                        a = a @ W[2 * l].T + W[2 * l + 1]
                        a = _gelu(a) if l < 3 else a
                    out.append(torch.exp(data.tmu + data.tsd * a) - 1)
                return torch.cat(out)

            sea.net = net
        if c["kind"] != "ensemble" and w.forced:
            following = w.next
            if w.storm:
                m, n = np.meshgrid(np.arange(w.kw["mm"]), np.arange(w.kw["nm"]), indexing="ij")
                u, v = _holland(m * c["dx"], n * c["dx"], w.storm)
                following = dict(uw=u, vw=v)
            sea.level(following)
        names = MEMBER_FIELDS if c["kind"] == "ensemble" else POINT_FIELDS
        if c["kind"] == "cycle":
            rng = np.random.default_rng([int(seed), 3])
            sea.e *= _tensor(rng.uniform(0.9, 1.1, size=(sea.n, 1, 1)))[:, 0, 0]
            names = ("ustar", "ht")
        if c["kind"] == "operators":
            s = 0.0
            while s < c["dtg"]:
                old, sea_ustar = sea.e.clone(), sea.ustar
                s += sea.substep(s)
            new, ustar, sea.e, sea.ustar = sea.e, sea.ustar, old, sea_ustar
            got = sea.sources(sea.oc)
            sea.e, sea.ustar = new, ustar
            sea.ocean(got)
            names = names + OCEAN_FIELDS
        else:
            sea.run_dtg()
        sea.stokes()
        sea.diag()
        out = {n: getattr(sea, n) for n in names}
        if c["profile"]:
            out.update(us=sea.us, vs=sea.vs)
        if c["kind"] == "cycle":
            out["e"] = sea.e.permute(2, 1, 0).contiguous()
        outs.append(out)
    return outs if c["kind"] == "ensemble" else outs[0]
