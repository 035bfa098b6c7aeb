"""The launch shapes of the tunable kernels: what the autotuner times and
picks, and that no shape changes a result."""
import pytest

import epic_amd as ea
from tests.gpu_util import say

pytestmark = pytest.mark.gpu

# the default operators, and the ones with kernels of their own: del^8 after
# del^4's pieces, monotonized fourth-order advection of every field
PLAIN = ea.spec(ea.JUPITER_LIKE, 64, 32, 20, 60, 5, 0.5, 0.0, 0.0, 0.5)
OTHER = ea.spec(ea.JUPITER_LIKE, 64, 32, 20, 60, 6, 0.0, 0.0, 0.0, 0.5, nu8=0.5, adv_mass=1, adv_nonmass=1)


def engine(*specs, precision=ea.FP64):
    e = ea.Engine(precision, len(specs))
    for sp in specs:
        e.add(sp)
    return e


def report(e):
    """{knob: what the autotuner says of it} of a one-bucket engine."""
    rep = e.autotune(1)
    say(rep)
    return dict(line.split(" ", 2)[2].split("=", 1) for line in rep.strip().splitlines())


def test_a_knob_no_launch_reads_stays_as_it_was():
    """del^4 alone runs in k_hv4 and the predictor-corrector's column pass in
    registers: neither reads rows_zhv, rows_d2 or cols_hsuv.  Set by hand or
    not, these stay, and the report says why."""
    say("knobs not launched")
    e = engine(PLAIN)
    e.set_shape("rows_zhv", 8)
    got = report(e)
    assert got["rows_zhv"] == "8 (not launched)"
    assert got["rows_d2"] == got["cols_hsuv"] == "built-in (not launched)"
    e.close()


def test_every_knob_is_timed_on_the_kernels_that_read_it():
    say("knobs launched")
    e = engine(OTHER)
    got = report(e)
    assert sorted(got) == sorted(ea.SHAPE_KNOBS)
    for k, v in got.items():
        assert v.endswith(" us/step)") and "(0.0 " not in v, (k, v)
    e.close()


@pytest.mark.parametrize("precision", [ea.FP64, ea.MIXED])
@pytest.mark.parametrize("knob", ["cols_p2etc", "cols_gz3", "cols_calcw"])
def test_the_widest_column_tile_fits_the_deepest_grid(knob, precision):
    """64 columns of 64 levels are one LDS array of 33 KB, and the built-in
    tile of a deep grid: the same shape by hand gives the same bits."""
    sp = ea.spec(ea.HELD_SUAREZ, 16, 8, 64, 300, 3, 0.5, 0.0, 0.1, 0.3)
    say("64 columns of 64 levels", knob, precision)
    out = []
    for v in (0, 64, 2064, 4064):
        e = engine(sp, precision=precision)
        e.set_shape(knob, v)
        e.step(3)
        out.append({f: e.read(0, f).tobytes() for f in ea.FIELDS if f[:4] not in ("DUDT", "DVDT")})
        e.close()
    for got in out[1:]:
        assert got == out[0]


def test_shapes_belong_to_buckets_of_the_same_kernels():
    """A shape chosen for a bucket serves later buckets of the grid, member
    count, hyperviscosity order and advection schemes it was chosen for, and
    no other: here the report of knobs that no launch of the new bucket reads
    shows what they hold."""
    say("shapes of other kernels")
    e = engine(OTHER)
    e.set_shape("cols_hsuv", 2016)
    e.set_shape("rows_zhv", 8)
    e.remove(0)
    e.add(PLAIN)
    got = report(e)
    assert got["cols_hsuv"] == got["rows_zhv"] == "built-in (not launched)"
    e.close()
    e = engine(PLAIN)
    e.set_shape("rows_zhv", 8)
    e.remove(0)
    e.add(PLAIN)
    assert report(e)["rows_zhv"] == "8 (not launched)"
    e.close()


def test_the_report_names_the_threads_that_are_launched():
    """set_p2etc, gz3 and calc_w give a thread 2, 4 or 8 of a column's 20
    levels (10, 5 or 3 threads a column); the Akima column pass has 256, 512 or
    1024 threads, or one for each of 22 levels."""
    say("threads in the report")
    e = engine(OTHER)
    for knob, text in report(e).items():
        if not knob.startswith("cols_") or text.startswith("built-in"):
            continue
        c, threads = text.split()[0].removesuffix("thr").split("/")
        c, threads = int(c), int(threads)
        if knob == "cols_hsuv":
            assert threads in (256, 512, 1024, 22 * c), (knob, text)
        else:
            assert threads in (10 * c, 5 * c, 3 * c), (knob, text)
    e.close()


# 35 rows (36 on the v grid) and 13 levels: a remainder over every tile
ODD = dict(ni=64, nj=34, nk=13, dt=60)
BY_KERNEL = {
    # the Akima scheme's column pass and its meridional tile
    "akima_cols": ("cols_hsuv", (16, 32, 64, 2032, 4064, 10004, 10012), dict(adv_mass=1, adv_nonmass=1)),
    "akima_rows": ("rows_mer", (2, 4, 8), dict(adv_mass=1, adv_nonmass=1)),
    # the predictor-corrector's meridional pass, a template instance each
    "hsu_rows": ("rows_mer", (2, 4, 8), {}),
    # the separate hyperviscosity kernels, which orders past del^4 take
    "del8_zonal": ("rows_zhv", (4, 8, 16), dict(nu4=0.0, nu8=0.5)),
    "del8_meridional": ("rows_d2", (8, 16, 32), dict(nu4=0.0, nu8=0.5)),
    "del6_zonal": ("rows_zhv", (4, 8, 16), dict(nu4=0.25, nu6=0.2)),
}


@pytest.mark.parametrize("precision", [ea.FP64, ea.MIXED])
@pytest.mark.parametrize("name", sorted(BY_KERNEL))
def test_every_shape_of_a_kernel_gives_the_same_bits(name, precision):
    """Each candidate on a member whose step launches the kernel that reads
    it (the report's time shows that it does)."""
    knob, values, opt = BY_KERNEL[name]
    sp = ea.spec(ea.JUPITER_LIKE, ODD["ni"], ODD["nj"], ODD["nk"], ODD["dt"], seed=9,
                 **dict(dict(nu4=0.5, noise_theta=0.0, noise_uv=0.5), **opt))
    e = engine(sp, precision=precision)
    assert report(e)[knob].endswith(" us/step)")
    e.close()
    out = {}
    for v in (0,) + values:
        say(name, precision, v)
        e = engine(sp, precision=precision)
        e.set_shape(knob, v)
        e.step(3)
        out[v] = {f: e.read(0, f).tobytes() for f in ea.FIELDS if f[:4] not in ("DUDT", "DVDT")}
        e.sync()
        e.close()
    bad = [(v, f) for v in values for f in out[0] if out[v][f] != out[0][f]]
    assert not bad
