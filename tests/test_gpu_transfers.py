"""Spectra and Stokes profiles on their way to and from the host: what is set
is what is read, over the sizes where the staged transfers change."""
import ctypes as C
import os

import numpy as np
import pytest

from umwm_amd import build, configs, hip

pytestmark = pytest.mark.gpu


def domain(mm, nm, om, pm, precision):
    wl = configs.regional_random(5, mm, nm, om, pm, dx=8e3, land_frac=0.1, shelf=True, wspd=14.0)
    d = hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=precision)
    d.init_jonswap(wl.jonswap)
    d.stokes_drift(True)
    return d


# one workgroup of points and rows that leave a remainder; several; more
# points than the staging holds (32 MiB), none a multiple of 64
@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("grid", [(6, 5, 25, 24), (14, 13, 37, 36), (83, 71, 31, 44)])
def test_spectra_round_trip(grid, precision):
    d = domain(*grid, precision)
    try:
        rng = np.random.default_rng(1)
        x = rng.uniform(0.0, 2.0, size=(d.im, d.pm, d.om))
        x[rng.uniform(size=x.shape) < 0.05] = 0.0
        if precision == 4:
            x = x.astype(np.float32).astype(np.float64)
        for name in ("e", "ef"):
            d.set(name, x)
            np.testing.assert_array_equal(d.get(name), x)
        # a point's bins reach that point: one point's spectrum set to zero
        # takes the wave height of that point and no other's
        d.diag()
        ht = d.get("ht")
        q = d.im - 1
        x[q] = 0.0
        d.set("e", x)
        d.diag()
        now = d.get("ht")
        assert now[q] == 0.0 and ht[q] > 0.0
        np.testing.assert_array_equal(now[:q], ht[:q])
    finally:
        d.close()


# more values than the staging holds, and fewer
@pytest.mark.parametrize("grid", [(13, 12), (352, 341)])
def test_stokes_rows(grid):
    d = domain(*grid, 25, 24, 4)
    try:
        us, vs = d.get("us"), d.get("vs")
        speed = np.hypot(us, vs)
        assert speed.shape == (d.lm, d.im) and np.all(speed[0] > 0.0)
        # the drift of a JONSWAP sea falls with depth at each point, and its
        # direction is the same at all levels to rounding: rows out of place
        # would show at points of other depths and winds
        assert np.all(speed[1:] <= speed[:-1] * (1 + 1e-6))
        assert np.all(np.abs(us[1:] * vs[:1] - vs[1:] * us[:1]) <= 0.2 * speed[1:] * speed[:1])
    finally:
        d.close()


def free_bytes():
    hiprt = C.CDLL(os.path.join(build.ROCM, "lib", "libamdhip64.so"))
    free, total = C.c_size_t(), C.c_size_t()
    assert hiprt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("precision", [8, 4])
def test_transfers_allocate_nothing(precision):
    """What get and set need on the device comes with the domain: a program
    that reads and sets fields between substeps_noalloc calls allocates none."""
    def transfers(d):
        e = d.get("e")
        d.set("e", e)
        d.get("us")

    d = domain(14, 13, 37, 36, precision)
    transfers(d)  # the runtime's own first use
    big = domain(83, 71, 31, 44, precision)
    try:
        before = free_bytes()
        transfers(big)
        assert free_bytes() == before
    finally:
        d.close()
        big.close()
