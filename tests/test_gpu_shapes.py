"""The launch shapes the fused kernels choose for default tiles (frequency
chunks, directions per wave, split advection) against the same substeps under
an explicit tile, at the sizes where the choice changes; and the directional
moments formed after a spectrum is set against those the advection leaves."""
import numpy as np
import pytest

from umwm_amd import autotune, configs, hip

pytestmark = pytest.mark.gpu

# (mm, nm, om, pm): two directions a wave and the most chunks; one point block
# with idle lanes; pm = 28 (no divisor 9 or 6); pm = 44 and 68 (one direction
# segment, prime pm / 4); pm = 48; chunks that do not divide om; one chunk;
# a spectrum wider than the split takes
GRIDS = [(12, 11, 37, 36), (5, 4, 25, 24), (30, 21, 31, 28), (30, 20, 26, 44), (16, 14, 33, 68),
         (60, 45, 41, 48), (105, 101, 29, 36), (190, 170, 25, 24), (14, 12, 25, 76)]


def fresh(grid, precision):
    mm, nm, om, pm = grid
    wl = configs.regional_random(7, mm, nm, om, pm, dx=1e4, land_frac=0.1, shelf=True, wspd=11.0,
                                 wdir=0.4)
    d = hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=precision)
    d.init_jonswap(wl.jonswap)
    d.stokes_drift(True)
    return d


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("grid", GRIDS)
def test_default_shape_equals_explicit_tile(grid, precision):
    # the same operations in the same order per bin; the rates of an explicit
    # tile with an even D are paired, which regroups one sum: a few ulp
    tol = 1e-13 if precision == 8 else 1e-5
    pm = grid[3]
    a, b = fresh(grid, precision), fresh(grid, precision)
    try:
        D = 9 if pm <= 72 else 18
        b.set_tile(D, -(-pm // D), D, -(-pm // D), 2)
        for n in (1, 3):
            ra, rb = a.substeps(n), b.substeps(n)
            assert ra[2] == rb[2] and abs(ra[1] - rb[1]) <= tol * abs(rb[1])
        for name in ("e", "ustar", "physics_time_step"):
            x, y = a.get(name), b.get(name)
            assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y), name
        dts = min(float(a.get("physics_time_step").min()), a.scalar("dtamin"))
        assert a.scalar("dts") == dts
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("grid", [(12, 11, 37, 36), (30, 21, 31, 28), (105, 101, 29, 24)])
def test_moments_after_set_equal_advection(grid, precision):
    """Setting the spectrum to itself makes the next substep form the moments
    anew: what the advection had left.  FP64 agrees bit for bit; in FP32 the
    host may flush subnormal bins (below 1.2e-38) on the way through set, so
    the spectra agree to far below the rounding of a different sum."""
    a, b = fresh(grid, precision), fresh(grid, precision)
    try:
        for d in (a, b):
            d.substeps(3)
        e = b.get("e")
        b.set("e", e)
        a.substeps(2)
        b.substeps(2)
        tol = 0.0 if precision == 8 else 1e-12
        for name in ("e", "ustar"):
            x, y = a.get(name), b.get(name)
            assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y), name
    finally:
        a.close()
        b.close()


def wide(dx, precision, pm=36, currents=False):
    wl = configs.tiny(3, 145, 140, 25, pm, winds=True, currents=currents, wspd=14.0)
    wl.params.delx = wl.params.dely = dx
    wl.params.dtg = 900.0
    d = hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=precision)
    d.init_jonswap(wl.jonswap)
    d.stokes_drift(True)
    d.forcinginput(wl.forcing_input(1))
    return d


# substeps whose sources are integrated ahead of their rates, where the
# advective limit holds throughout (1 km), where the sources' time scales hold
# (30 km) and where both do in turn, against the plain order of an explicit
# tile: the same lengths, the same state to rounding
@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("dx,pm,currents", [(1e3, 36, False), (6e3, 36, False), (9e3, 24, False),
                                            (12e3, 28, False), (3e4, 36, False), (1e3, 36, True)])
def test_sources_ahead_of_rates(dx, pm, currents, precision):
    tol = 1e-12 if precision == 8 else 1e-5
    a, b = wide(dx, precision, pm, currents), wide(dx, precision, pm, currents)
    try:
        D = 6 if pm == 24 else 9
        b.set_tile(D, -(-pm // D), 18, -(-pm // 18), 2)  # 18 directions: never ahead
        for k in range(12):
            ra, rb = a.substep(), b.substep()
            assert abs(ra[1] - rb[1]) <= tol * rb[1], (k, ra, rb)
            assert abs(ra[0] - rb[0]) <= tol * rb[0], (k, ra, rb)
        pts = a.get("physics_time_step")
        assert np.allclose(pts, b.get("physics_time_step"), rtol=10 * tol, atol=0)
        assert a.scalar("dts") <= float(pts.min()) * (1 + tol)
        na, nb = a.run_dtg(), b.run_dtg()  # the rest of a window, and its short last substep
        na, nb = a.run_dtg(), b.run_dtg()
        assert na == nb and a.scalar("sumt") == b.scalar("sumt") == 900.0
        for name in ("e", "ustar", "ht", "cd"):
            x, y = a.get(name), b.get(name)
            assert np.linalg.norm(x - y) <= 10 * tol * np.linalg.norm(y), name
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("precision", [8, 4])
def test_sources_ahead_with_a_given_tile(precision):
    tol = 1e-12 if precision == 8 else 1e-5
    a, b = wide(1e3, precision), wide(1e3, precision)
    try:
        a.set_tile(18, 2, 9, 4, 2)
        b.set_tile(18, 2, 18, 2, 2)
        assert a.run_dtg() == b.run_dtg()
        for name in ("e", "ustar", "physics_time_step"):
            x, y = a.get(name), b.get(name)
            assert np.linalg.norm(x - y) <= 10 * tol * np.linalg.norm(y), name
    finally:
        a.close()
        b.close()


def test_sources_ahead_in_a_batch():
    """Members that run ahead beside members that may not (currents) or cannot
    (their time scales): each as by itself."""
    spec = [(1e3, False), (1e3, True), (3e4, False)]
    one = [wide(dx, 8, 36, c) for dx, c in spec]
    many = [wide(dx, 8, 36, c) for dx, c in spec]
    batch = hip.Batch(many)
    try:
        for _ in range(2):
            batch.run_dtg()
            for x in one:
                x.run_dtg()
        for x, y in zip(one, many):
            for name in ("e", "ustar", "ht"):
                u, v = x.get(name), y.get(name)
                assert np.linalg.norm(u - v) <= 1e-12 * np.linalg.norm(v), name
    finally:
        batch.close()
        for x in one + many:
            x.close()


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("om,pm", [(6, 16), (7, 4), (5, 36), (7, 28)])
def test_few_frequencies(om, pm, precision):
    """One chunk of two directions a wave on a small grid: a shape whose sources
    are not integrated ahead, over substeps that the advective limit holds."""
    wl = configs.tiny(4, 16, 13, om, pm, wspd=14.0)
    wl.params.delx = wl.params.dely = 300.0
    a, b = (hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=precision)
            for _ in range(2))
    try:
        D = 6 if pm % 6 == 0 else 9
        b.set_tile(D, -(-pm // D), D, -(-pm // D), 2)
        for d in (a, b):
            d.init_jonswap(wl.jonswap)
            d.stokes_drift(True)
            d.substeps(12)
        tol = 1e-12 if precision == 8 else 1e-5
        for name in ("e", "es", "ustar"):
            x, y = a.get(name), b.get(name)
            assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y), name
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("precision", [8, 4])
def test_lengths_kept_or_left_to_the_rates(precision):
    """The third substep's time scales against the advective limit it was
    guessed to take: below it (the guess is taken back), within the hundredth
    that the sources' rounding is given (left to the rates) and above it (kept).
    The guesses are counted, and the lengths are those of the plain order, bit
    for bit.  With currents no guess is made."""
    tol = 1e-12 if precision == 8 else 1e-5

    def start(explim=None, currents=False):
        wl = configs.tiny(3, 145, 140, 25, 36, winds=True, currents=currents, wspd=14.0)
        wl.params.delx = wl.params.dely = 1e3
        wl.params.dtg = 900.0
        if explim:
            wl.params.explim = explim
        d = hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=precision)
        d.init_jonswap(wl.jonswap)
        d.stokes_drift(True)
        d.forcinginput(wl.forcing_input(1))
        return d, wl.params.explim

    d, explim = start()
    d.substeps(3)
    # the limit holds throughout, so that the state does not depend on explim
    limit = float(d.get("physics_time_step").min()) / d.scalar("dtamin")
    assert limit > 2 and d.scalar("dts") == d.scalar("dtamin")
    d.close()
    for ratio, ahead, missed in ((0.97, 1, 1), (1.005, 1, 1), (1.5, 2, 0)):
        a, b = (start(explim * ratio / limit)[0] for _ in range(2))
        try:
            b.set_tile(9, 4, 18, 2, 4)  # never ahead
            for k in range(3):
                assert a.substep() == b.substep(), (ratio, k)
                assert a.scalar("dts") == b.scalar("dts")
            assert (a.scalar("dts") == a.scalar("dtamin")) == (ratio > 1)
            assert a.scalar("substeps_ahead") == ahead, ratio
            assert a.scalar("substeps_missed") == missed, ratio
            assert b.scalar("substeps_ahead") == b.scalar("substeps_missed") == 0
            for name in ("e", "ustar", "physics_time_step", "wspd", "shelt", "oc"):
                x, y = a.get(name), b.get(name)
                assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y), (ratio, name)
        finally:
            a.close()
            b.close()
    d, _ = start(currents=True)
    d.substeps(4)
    assert d.scalar("substeps_ahead") == d.scalar("substeps_missed") == 0
    d.close()


@pytest.mark.parametrize("grid", [(270, 250, 7, 28), (270, 250, 6, 32), (190, 180, 7, 68),
                                  (250, 225, 6, 44)])
def test_nine_directions_with_idle_slots(grid):
    """FP32 grids large enough for waves of nine directions that do not divide
    pm, which run their sources ahead too: the bits of the plain order."""
    mm, nm, om, pm = grid
    wl = configs.tiny(4, mm, nm, om, pm, land=False, winds=True, wspd=14.0)
    wl.params.delx = wl.params.dely = 500.0
    a, b = (hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=4)
            for _ in range(2))
    try:
        assert (a.im + 63) // 64 * -(-pm // 9) >= 4096
        b.set_tile(9, -(-pm // 9), 9, -(-pm // 9), 4)  # never ahead
        for d in (a, b):
            d.init_jonswap(wl.jonswap)
            d.stokes_drift(True)
            d.forcinginput(wl.forcing_input(1))
        for _ in range(6):
            assert a.substep() == b.substep()
        assert a.scalar("substeps_ahead") > 0 and b.scalar("substeps_ahead") == 0
        for name in ("e", "es", "ustar"):
            assert np.array_equal(a.get(name), b.get(name)), name
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("grid", GRIDS)
def test_default_shape_equals_given_tile(grid, precision):
    """As test_default_shape_equals_explicit_tile, under a tile that is not the
    default and is therefore launched as it is given: the same bits."""
    pm = grid[3]
    a, b = fresh(grid, precision), fresh(grid, precision)
    try:
        D = 9 if pm <= 72 else 18
        b.set_tile(D, -(-pm // D), D, -(-pm // D), 4)
        assert b.tile()[4] == 4
        for n in (1, 3):
            assert a.substeps(n) == b.substeps(n)
        for name in ("e", "ustar"):
            assert np.array_equal(a.get(name), b.get(name)), name
    finally:
        a.close()
        b.close()


def test_the_default_tile_stands_for_the_choice():
    """Setting the tile that was read, or the default after another, leaves the
    launch shape to the grid, seen by the sources that run ahead with four
    directions a wave; a batch likewise."""
    doms = [wide(1e3, 8, 28) for _ in range(2)]
    d = doms[0]
    batch = hip.Batch(doms[1:])
    try:
        d.substeps(2)
        batch.substeps(2)

        def ahead(m, step):
            n = m.scalar("substeps_ahead")
            step(2)
            return m.scalar("substeps_ahead") - n

        assert d.tile() == autotune.default_tile(28) == (9, 4, 9, 4, 2)
        assert ahead(d, d.substeps) == 2
        d.set_tile(*d.tile())
        assert ahead(d, d.substeps) == 2
        d.set_tile(9, 4, 9, 4, 4)
        assert d.tile() == (9, 4, 9, 4, 4) and ahead(d, d.substeps) == 0
        d.set_tile(*autotune.default_tile(28))
        assert ahead(d, d.substeps) == 2
        m = doms[1]
        assert ahead(m, batch.substeps) == 2
        batch.set_tile(9, 4, 18, 2, 2)
        assert ahead(m, batch.substeps) == 0
        batch.set_tile(*autotune.default_tile(28))
        assert ahead(m, batch.substeps) == 2
    finally:
        batch.close()
        for x in doms:
            x.close()


def test_autotune_keeps_the_default_where_it_is_faster():
    """On a small grid the shape split over frequency chunks takes half the
    time of any tile, whose kernels the tuner times one by one."""
    d = fresh((64, 48, 37, 36), 8)
    try:
        d.substeps(3)
        choice, table = autotune.autotune(d, steps=3)
        assert choice == d.tile() == autotune.default_tile(36) and len(table) == 4
    finally:
        d.close()


@pytest.mark.parametrize("grid", [(270, 250, 6, 36), (190, 180, 7, 72)])
def test_rates_of_eighteen_directions(grid):
    """FP32 grids large enough for k_rates to take eighteen directions a wave,
    where the sources set the substep: the bits of nine."""
    mm, nm, om, pm = grid
    wl = configs.tiny(4, mm, nm, om, pm, land=False, winds=True, wspd=18.0)
    wl.params.delx = wl.params.dely = 2e5
    a, b = (hip.Domain(wl.params, wl.grid_input(), wl.forcing_input(0), precision=4)
            for _ in range(2))
    try:
        assert (a.im + 63) // 64 * (pm // 9) >= 4096
        b.set_tile(9, pm // 9, 18, pm // 18, 2)
        for d in (a, b):
            d.init_jonswap(wl.jonswap)
            d.stokes_drift(True)
            d.forcinginput(wl.forcing_input(1))
        for _ in range(4):
            assert a.substep() == b.substep()
        assert 0 < a.scalar("dts") < a.scalar("dtamin") and a.scalar("substeps_ahead") == 0
        for name in ("physics_time_step", "e", "ustar"):
            assert np.array_equal(a.get(name), b.get(name)), name
    finally:
        a.close()
        b.close()
