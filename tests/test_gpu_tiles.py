"""The step's register tiles at their edges: every field bit for bit against
the oracle with the GPU's exp, log and pow (the FP64 kernels perform its
operations in its order, so the tolerance is zero) after the Adams-Bashforth
start-up and one third-order step."""
import pytest

import epic_amd as ea
from oracle.cpuref import CpuRef
from tests.gpu_util import bitwise_diff, say

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
