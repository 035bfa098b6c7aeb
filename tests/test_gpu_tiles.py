"""The step's register tiles at their edges: every field bit for bit against
the oracle with the GPU's exp, log and pow (the FP64 kernels perform its
operations in its order, so the tolerance is zero) after the Adams-Bashforth
start-up and one third-order step."""
import numpy as np
import pytest

import epic_amd as ea
from oracle.cpuref import CpuRef
from tests.gpu_util import FLOOR_FACTOR, bitwise_diff, say

pytestmark = pytest.mark.gpu

# planet, ni, nj, nk, dt, options.  Rows nj+1 leave 0-3 over a meridional tile
# of 4 and 1-7 over one of 8; nk leaves every remainder of 2, 4 and 8 levels
# per lane; ni = 8 is the shortest row (many rows per wavefront), 32 has rows
# that share a wavefront, 64 the first with a wavefront (and scalar rows) of
# its own, 512 a block of its own.
TILES = {
    "shortest": (ea.HELD_SUAREZ, 8, 6, 4, 600, {}),
    "rows_share_a_wavefront": (ea.VENUS_LIKE, 32, 17, 5, 300, {}),
    "one_row_over": (ea.JUPITER_LIKE, 64, 32, 7, 60, {}),
    "two_rows_over": (ea.SATURN_LIKE, 64, 33, 9, 60, {}),
    "three_rows_over": (ea.HOT_JUPITER, 64, 34, 13, 30, {}),
    "two_levels_per_lane": (ea.JUPITER_LIKE, 128, 21, 11, 60, {}),
    # (62 rows are too few for 512 columns: the oracle's third step is not
    # monotone any more, and the engine must say so too)
    "wide_rows": (ea.JUPITER_LIKE, 512, 62, 5, 30, {}),
    "wide_rows_stable": (ea.JUPITER_LIKE, 512, 126, 5, 30, {}),
    "four_levels_per_lane": (ea.JUPITER_LIKE, 256, 66, 18, 30, {}),
    # 4.3 million points in the bucket: 8 levels and rows per lane throughout
    "eight_levels_per_lane": (ea.JUPITER_LIKE, 128, 32, 9, 60, dict(members=112)),
    "averaged_pv": (ea.JUPITER_LIKE, 64, 18, 6, 60, dict(pv_scheme=1)),
    "winds_in_place": (ea.HELD_SUAREZ, 32, 19, 6, 300, dict(nu6=0.2)),
    "no_hyperviscosity": (ea.JUPITER_LIKE, 32, 15, 8, 60, dict(nu4=0.0)),
    "schemes_differ": (ea.JUPITER_LIKE, 64, 22, 10, 60, dict(adv_nonmass=1)),
}


@pytest.mark.parametrize("name", sorted(TILES))
def test_tile_edges_equal_the_oracle(name):
    planet, ni, nj, nk, dt, opt = TILES[name]
    opt = dict(opt)
    members, nu4 = opt.pop("members", 1), opt.pop("nu4", 0.4)
    specs = [ea.spec(planet, ni, nj, nk, dt, 41 + m, nu4, 0.1, 0.3, 0.5, **opt) for m in range(members)]
    say("tile", name, ni, nj, nk, members)
    eng = ea.Engine(ea.FP64, members)
    try:
        slots = [eng.add(sp) for sp in specs]
        eng.step(3)
        try:
            eng.sync()
            fatal = False
        except ea.EpicError:
            fatal = True
        for m in {0, members - 1}:
            ref = CpuRef(specs[m], nudged="cr")
            ref.sync()
            assert (ref.step(3) != 0) == fatal, (name, m)
            bad = [] if fatal else bitwise_diff(lambda f: eng.read(slots[m], f), ref.read)
            ref.close()
            assert not bad, (name, m, bad)
    finally:
        eng.close()


def rounded_oracle(sp, fields):
    """The oracle's fields after three steps with h and theta moved by up to
    2^-24 of themselves after each."""
    r, rng = CpuRef(sp, nudged="cr"), np.random.default_rng(1)
    r.sync()
    for _ in range(3):
        assert r.step(1) == 0
        for f in ("HDRY", "THETA"):
            x = r.read(f)
            e = 1. + 2. ** -24 * rng.uniform(-1., 1., x.shape)
            e[:, :, 0], e[:, :, -1] = e[:, :, -2], e[:, :, 1]
            r.write(f, x * e)
    out = {f: r.read(f) for f in fields}
    r.close()
    return out


@pytest.mark.parametrize("name", sorted(set(TILES) - {"wide_rows"}))
def test_mixed_tile_edges_follow_the_oracle(name):
    """The FP32 instances of the same tiles.  A field's change over a step
    goes through FP32 once (advection, hyperviscosity in two directions,
    momentum terms), and is at most the field itself: a few roundings of 2^-24
    a step, so 1e-6 of the largest value of h, theta and p after three steps.
    The winds also answer to the errors of h and theta through the pressure
    gradient: 1e-5 of the fastest wind (not on the hot Jupiter, whose winds
    start at rest).  Where the grid itself amplifies them (of 128 columns and
    22 rows the fastest wind grows by a third in the three steps) it is ten
    times what one FP32 rounding a step of the oracle's own h and theta does to
    its fields.  A member of many has the bits it has alone, where its tiles
    are smaller."""
    planet, ni, nj, nk, dt, opt = TILES[name]
    opt = dict(opt)
    members, nu4 = opt.pop("members", 1), opt.pop("nu4", 0.4)
    specs = [ea.spec(planet, ni, nj, nk, dt, 41 + m, nu4, 0.1, 0.3, 0.5, **opt) for m in range(members)]
    say("mixed tile", name, ni, nj, nk, members)
    eng = ea.Engine(ea.MIXED, members)
    try:
        for sp in specs:
            eng.add(sp)
        eng.step(3)
        eng.sync()
        for m in {0, members - 1}:
            ref = CpuRef(specs[m], nudged="cr")
            ref.sync()
            assert ref.step(3) == 0
            got = {f: eng.read(m, f) for f in ("U", "V", "HDRY", "THETA", "P3")}
            want = {f: ref.read(f) for f in got}
            ref.close()
            wind = max(abs(want["U"]).max(), abs(want["V"]).max())
            floor = rounded_oracle(specs[m], got)
            for f, a in got.items():
                if f in ("U", "V") and planet == ea.HOT_JUPITER:
                    continue
                scale, tol = (wind, 1e-5) if f in ("U", "V") else (abs(want[f]).max(), 1e-6)
                tol = max(tol, FLOOR_FACTOR * float(abs(floor[f] - want[f]).max() / scale))
                worst = float(abs(a - want[f]).max() / scale)
                say(f, m, f"{worst:.1e} of the largest")
                assert worst <= tol, (name, m, f, worst)
            if members > 1:
                alone = ea.Engine(ea.MIXED, 1)
                alone.add(specs[m])
                alone.step(3)
                assert not bitwise_diff(lambda f: eng.read(m, f), lambda f: alone.read(0, f), sorted(got))
                alone.close()
    finally:
        eng.close()
