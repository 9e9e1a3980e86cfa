"""Stokes drift, diag and the ice wave height at the sizes where their kernel's
shape changes, against plain FP64 sums over the spectrum the domain holds."""
import numpy as np
import pytest

from umwm_amd import abi, configs, hip

pytestmark = pytest.mark.gpu


def fresh(mm, nm, om, pm, precision, depths, shelf=True):
    wl = configs.regional_random(11, mm, nm, om, pm, dx=1e4, land_frac=0.1, shelf=shelf,
                                 wspd=13.0, wdir=0.7)
    if depths is not None:
        wl.params.depths[:] = list(depths) + [-1.0] * (100 - len(depths))
    d = hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=precision)
    d.init_jonswap(wl.jonswap)
    return wl, d


def reference(d, wl):
    """us, vs, ht, mwp, mss, dominant bin from the domain's e and tables."""
    e = d.get("e").transpose(2, 1, 0)  # (om, pm, im)
    k, kdk, dwn = d.get("k").T, d.get("kdk").T, d.get("dwn").T
    om, pm = e.shape[:2]
    p = wl.params
    f = np.exp(np.log(p.fmin) + np.arange(om) * (np.log(p.fmax) - np.log(p.fmin)) / (om - 1))
    dth = 2 * np.pi / pm
    th = (np.arange(1, pm + 1) - 0.5 * (pm + 1)) * dth
    a = (e * np.cos(th)[None, :, None]).sum(1)
    b = (e * np.sin(th)[None, :, None]).sum(1)
    dj = d.get("d")[: d.im]
    us, vs = [], []
    for depth in [q for q in p.depths if q >= 0]:
        arg, kd = 2 * k * (dj - depth), k * dj
        deep = (np.abs(arg) > 50) | (kd > 50)
        with np.errstate(over="ignore"):
            t = np.where(deep, 2 * np.exp(-2 * k * depth), np.cosh(np.minimum(arg, 50)) / np.sinh(np.minimum(kd, 50)) ** 2)
        t = np.where(depth > dj, 0.0, 2 * np.pi * f[:, None] * k ** 2 * t * dwn * dth)
        us.append((t * a).sum(0))
        vs.append((t * b).sum(0))
    s = e.sum(1) * kdk
    m0, m2, mk = s.sum(0), (f[:, None] ** 2 * s).sum(0), (s * k ** 2).sum(0)
    top = (e * kdk[:, None, :]).transpose(1, 0, 2).reshape(om * pm, -1).argmax(0)
    return dict(us=np.array(us), vs=np.array(vs), ht=4 * np.sqrt(m0 * dth), mwp=np.sqrt(m0 / m2),
                mss=mk * dth, dwp=1 / f[top % om], dwd=th[top // om])


# (mm, nm): one pass for both operators; 16 points a workgroup; 64 points a
# workgroup; level lists: one, the default 42, 49 (a second level group), 100
@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("grid,levels", [((9, 8, 25, 24), 1), ((12, 11, 37, 36), None),
                                         ((40, 33, 29, 28), 100), ((120, 100, 26, 28), 49),
                                         ((200, 190, 25, 24), None), ((190, 180, 25, 24), 100)])
def test_integrals_against_fp64_sums(grid, levels, precision):
    depths = None if levels is None else np.linspace(0.1, 400.0, levels)
    wl, d = fresh(*grid, precision, depths)
    try:
        d.stokes_drift(True)
        d.diag()
        ref = reference(d, wl)
        # FP64 sums of the same e and tables, which the FP32 domain holds in
        # FP32: k there is rounded, and e^{2kz} carries 2kz ulps of it
        for name, want in ref.items():
            got = d.get(name)
            tol = 1e-12 if precision == 8 else 1e-4
            assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), name
        # the ice wave height follows a set spectrum
        e = d.get("e")
        d.set("e", e)
        assert np.linalg.norm(d.get("hs_ice") - ref["ht"]) <= 1e-6 * np.linalg.norm(ref["ht"])
        both = {n: d.get(n) for n in ("us", "vs", "ds", "ht", "mwd", "dwp")}
        d.substeps(2)
        d.set("e", e)
        d.stokes_drift()
        d.diag()
        for n, v in both.items():
            assert np.array_equal(d.get(n), v), n
    finally:
        d.close()
