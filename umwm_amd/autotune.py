"""Tile-shape autotuner for the fused kernels.

k_rates and k_integrate give each thread D consecutive directions of one
sea point and W = ceil(pm / D) waves per workgroup; k_advect keeps NB
directions of gathers in flight per wave.  Larger D means that a
frequency's tables are formed for more directions at once but more
registers; larger NB means more loads in flight but fewer resident waves.
The best shape depends on pm, the precision and the grid size, so it is
measured: each candidate runs a few live substeps with HIP-event timing
and the fastest shape per kernel is kept.  Whole substeps then decide
between that tile and the default one, which splits the sweeps of small
grids over frequency and integrates the sources ahead of their rates where
it can, neither of which the kernels' own times show.  Candidates only
change the order of directional sums, so the model state advances normally
while tuning.
"""
import math
import time

RATES_D = (6, 9, 18, 36)
INTEGRATE_D = (3, 6, 9, 12, 18)
ADVECT_NB = (2, 4)


def candidates(pm, ds):
    out = []
    for D in ds:
        W = math.ceil(pm / D)
        if 1 <= W <= 8:
            out.append((D, W))
    return out


def default_tile(pm):
    """The tile of a new domain, which stands for a launch shape by the size
    of its grid (umwm_hip_set_tile)."""
    def first(ds):
        return next((D, math.ceil(pm / D)) for D in ds if math.ceil(pm / D) <= 8)
    return first((9, 18, 36)) + first((9, 12, 18, 36)) + (2,)


def substep_time(dom, tile, steps):
    """Seconds of a live substep under `tile`, back to back; None where the
    time of the forcing window ran out meanwhile (what is left does nothing)."""
    dom.set_tile(*tile)
    dom.substeps(1)  # captures the launch
    n0 = dom.scalar("nsub")
    t0 = time.perf_counter()
    dom.substeps(steps)
    t = (time.perf_counter() - t0) / steps
    return t if dom.scalar("nsub") == n0 + steps else None


def autotune(dom, steps=3, verbose=None):
    """Chooses (D1, W1, D2, W2, NB) for `dom` by timing live substeps;
    returns the chosen tuple and the per-candidate mean kernel times (ms:
    rates, integrate, advect, stress)."""
    pm = dom.pm
    c1 = candidates(pm, RATES_D)
    c2 = candidates(pm, INTEGRATE_D)
    n = max(len(c1), len(c2), len(ADVECT_NB))
    table = []
    dom.set_timing(True)
    for k in range(n):
        a = c1[min(k, len(c1) - 1)]
        b = c2[min(k, len(c2) - 1)]
        nb = ADVECT_NB[min(k, len(ADVECT_NB) - 1)]
        dom.set_tile(a[0], a[1], b[0], b[1], nb)
        dom.timing(reset=True)
        for _ in range(steps):
            dom.substep()
        ms, cnt = dom.timing(reset=True)
        t = [m / max(c, 1) for m, c in zip(ms, cnt)]
        table.append((a, b, nb, t))
        if verbose:
            verbose(f"autotune: rates {a} integrate {b} advect NB={nb}: "
                    + ", ".join(f"{x:.3f}" for x in t) + " ms")
    dom.set_timing(False)
    best1 = min(c1, key=lambda a: min(t[0] for x, _, _, t in table if x == a))
    best2 = min(c2, key=lambda b: min(t[1] for _, y, _, t in table if y == b))
    best3 = min(ADVECT_NB, key=lambda nb: min(t[2] for _, _, z, t in table if z == nb))
    # whole substeps of the kernels' choice, of the same with the default's
    # k_integrate, and of the default: in turn, the faster of two passes each.
    # A later one has to be clearly faster: two that run their sources ahead
    # differ only in kernels that then do not run.  The default where nothing
    # could be timed.
    default = default_tile(pm)
    tiles = list(dict.fromkeys([best1 + best2 + (best3,), best1 + default[2:4] + (best3,), default]))
    times = [[substep_time(dom, x, steps) for x in tiles] for _ in range(2)]
    if all(t for row in times for t in row):
        best = [min(row[k] for row in times) for k in range(len(tiles))]
        k = 0
        for q in range(1, len(tiles)):
            if best[q] < 0.97 * best[k]:
                k = q
        choice = tiles[k]
        if verbose:
            verbose(f"autotune: substeps {dict(zip(tiles, best))} s, {choice}")
    else:
        choice = default
    dom.set_tile(*choice)
    return choice, table


def autotune_batch(batch, probe, steps=3, verbose=None):
    """Tunes a batch through one representative member `probe` (a Domain
    built like the largest member) and applies its choice to the batch."""
    choice, table = autotune(probe, steps=steps, verbose=verbose)
    batch.set_tile(*choice)
    return choice, table
