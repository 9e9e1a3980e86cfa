"""The operator kernels that give a wave a frequency, at the sizes where their
loops have remainders: against the FP64 CPU oracle, operator by operator."""
import numpy as np
import pytest

from umwm_amd import configs
from tests.harness import make_pair, relerr

pytestmark = pytest.mark.gpu

# (mm, nm, om, pm): fewer frequencies than waves; one frequency past the waves
# and directions that leave a partial group; more rows than the staged 64, with
# 130 points; fewer directions than one pass takes and one workgroup of lanes
GRIDS = [(9, 8, 5, 16), (14, 11, 17, 20), (16, 15, 33, 72), (10, 9, 16, 4)]


@pytest.mark.parametrize("ice", [False, True])
@pytest.mark.parametrize("grid", GRIDS)
def test_operators_by_rows(grid, ice, oracle_lib):
    mm, nm, om, pm = grid
    # sums of up to om * pm = 2,376 terms regrouped in FP64: 2,376 * 1.1e-16,
    # and a few ulp of each device function, stay below 1e-11 of the largest
    tol = 1e-11
    wl = configs.tiny(seed=3, mm=mm, nm=nm, om=om, pm=pm, winds=True, currents=True, ice=ice)
    o, d = make_pair(wl)
    try:
        for step in range(2):
            for name in ("forcinginterpolate", "sin_d12", "sds_d12", "snl_d12", "s_ice", "source",
                         "propagation", "refraction", "update"):
                getattr(o, name)()
                getattr(d, name)()
                fields = {"sin_d12": ["ssin"], "sds_d12": ["dummy", "sds"], "s_ice": ["sice"],
                          "source": ["ef"], "refraction": ["rotl", "rotr", "ef"],
                          "update": ["e"]}.get(name, [])
                for f in fields:
                    err = relerr(d.get(f), o.get(f))
                    assert err <= tol, (step, f, err)
            for s in ("dts", "dtr", "sumt"):
                assert abs(d.scalar(s) - o.scalar(s)) <= tol * max(abs(o.scalar(s)), 1.0), s
            o.stress_atm()
            d.stress("atm")
            o.stress_ocn()
            d.stress("ocn")
            for x, y in (("taux", "tauy"), ("taux_form", "tauy_form"),
                         ("taux_skin", "tauy_skin"), ("tailocnx", "tailocny"),
                         ("taux_ocntop", "tauy_ocntop"), ("taux_ocnbot", "tauy_ocnbot"),
                         ("taux_snl", "tauy_snl"), ("epsx_ocn", "epsy_ocn")):
                scale = max(np.max(np.abs(o.get(x))), np.max(np.abs(o.get(y))))
                for f in (x, y):
                    assert np.max(np.abs(d.get(f) - o.get(f))) <= tol * scale, (step, f)
            assert relerr(d.get("ustar"), o.get("ustar")) <= tol
            if step == 0:
                o.set_scalar("first", 0)
                d.end_first()
    finally:
        d.close()


@pytest.mark.parametrize("pm", [24, 28, 36, 72])
def test_wind_square_to_a_direction(pm, oracle_lib):
    """Winds along the axes, the diagonals and the directions themselves, some
    at a right angle to a bin, where the sign of cos(wdir - th) chooses between
    dissipation coefficients a hundredfold apart: each bin as the oracle has
    it."""
    # the wind input is a few products of values good to a few ulp (4e-15);
    # cancellation against the phase speed costs up to 1e-3 of that
    tol = 1e-11
    wl = configs.tiny(seed=5, mm=26, nm=24, om=25, pm=pm, land=False, winds=True)
    o, d = make_pair(wl)
    try:
        th = (np.arange(pm) + 1 - 0.5 * (pm + 1)) * (2 * np.pi / pm)
        diag = [np.arctan2(a, b) for a in (-1, 0, 1) for b in (-1, 0, 1) if a or b]
        wdir = np.resize(np.concatenate([diag, th, np.arange(-36, 37) * np.pi / 36]),
                         d.get("wdir").size)
        for m in (o, d):
            m.forcinginterpolate()
        d.set("wdir", wdir)
        o.raw("wdir")[1:] = wdir
        assert np.array_equal(d.get("wdir"), o.get("wdir"))
        d.sin_d12()
        o.sin_d12()
        x, y = d.get("ssin"), o.get("ssin")
        big = np.abs(y) > 1e-6 * np.max(np.abs(y), axis=(1, 2), keepdims=True)
        assert np.max(np.abs(x - y)[big] / np.abs(y[big])) <= tol
        assert relerr(x, y) <= tol
    finally:
        d.close()
        o.close()
