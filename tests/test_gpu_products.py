"""The NLL of products of 1-D leaves in logarithms (k_reduce_prod: flat trees at four events
per lane) against k_reduce_flat at two and the interpreter."""
import math

import numpy as np
import pytest

import oracle as O
from goofit_amd import capi

from _models import arrays

pytestmark = pytest.mark.gpu

OBS = [O.Obs(n, -10.0, 10.0, 50) for n in "wxyz"]


def _leaf(kind, obs, k):
    v = lambda name, x: O.Var(f"{name}{k}", x)
    if kind == "G":
        return O.Gaussian(f"g{k}", obs, v("m", 0.2 * k), v("s", 0.7 + 0.1 * k))
    if kind == "N":  # so narrow that most events underflow to 0 and some are subnormal
        return O.Gaussian(f"n{k}", obs, v("m", 0.0), v("s", 0.05))
    if kind == "E":
        return O.Exp(f"e{k}", obs, v("a", -0.4 - 0.1 * k))
    if kind == "X":
        return O.ExpGaus(f"x{k}", obs, v("xm", 0.1 * k), v("xs", 0.4), v("xr", 0.6))
    if kind == "U":  # exp(e) erfc(u) with erfc(u) rounded to 0 where exp(e) erfc(u) itself is not
        return O.ExpGaus(f"u{k}", obs, v("xm", 0.0), v("xs", 0.03), v("xr", 200.0))
    if kind == "P":  # exponents from -750 to 750
        return O.Exp(f"p{k}", obs, v("a", 250.0))
    if kind == "S":  # a negative width: erfc(u) the other way round, growing with x
        return O.ExpGaus(f"s{k}", obs, v("xm", 0.1 * k), v("xs", -0.4), v("xr", 0.6))
    return O.ExpGaus(f"z{k}", obs, v("xm", 0.0), v("xs", 0.4), v("xr", -0.6))  # a negative density


def _both(ctx):
    got = {}
    try:
        for knob in (4, 2, 0):
            ctx.set_tuning(capi.TUNE_FLAT, knob)
            got[knob] = ctx.reduce_metric("NLL")[0]
        for name, knob in ((capi.TUNE_FUSED_FINISH, 0), (capi.TUNE_INLINE_ARGS, 0)):
            ctx.set_tuning(capi.TUNE_FLAT, 4)
            ctx.set_tuning(name, knob)
            assert ctx.reduce_metric("NLL")[0] == got[4], name
            ctx.set_tuning(name, 1)
    finally:
        for name in (capi.TUNE_FLAT, capi.TUNE_FUSED_FINISH, capi.TUNE_INLINE_ARGS):
            ctx.set_tuning(name, 1)
    assert got[2] == got[0]
    return got[4], got[2]


@pytest.mark.parametrize("kinds", ["G", "X", "GEX", "XXGE", "GGEEXXGGEEXXGGEE", "GGEEXXGGEEXXGGEEX", "NG", "GZ", "U",
                                   "S", "GS", "P", "NP", "PGN"])
@pytest.mark.parametrize("n", [1, 255, 1025, 70_001])
def test_products_in_logarithms(ctx, kinds, n):
    """One leaf, one to four columns, two leaves on a column, the most leaves the kernel takes
    and one more, densities that underflow in some tiles or are negative (those events add 0 in
    the reference's metric), from one event to 69 workgroups with a ragged last tile.  Every
    event's logarithm carries a few roundings of its leaves' exponents on either path: 8 units of
    2^-53 of the exponents' sum for each, taken as if all had one sign."""
    rng = np.random.default_rng(n + len(kinds))
    cols = [rng.uniform(-3.0, 3.0, n) for _ in range(4)]
    ncols = min(len(kinds), 4)
    leaves = [_leaf(kind, OBS[k % 4], k) for k, kind in enumerate(kinds)]
    top = leaves[0] if len(leaves) == 1 else O.Prod("p", leaves)
    f, p, c, o, norms = arrays(top)[1]
    ctx.set_program(f, p, c, o, norms)
    ctx.upload_columns(cols[:ncols])
    ctx.update_norms(0.7 * np.asarray(norms, np.float64))
    log, plain = _both(ctx)
    exps = sum(0.5 * (x / s) ** 2 if s else np.abs(x) * (250 if "P" in kinds else 1) + (1500 if "U" in kinds else 12) for x, s in
               ((cols[k % 4], {"G": 0.7, "N": 0.05}.get(kind)) for k, kind in enumerate(kinds)))
    if "P" in kinds and math.isinf(plain):
        assert log == plain
        return
    assert math.isfinite(log)
    assert abs(log - plain) <= 16 * 2.0**-53 * (np.sum(np.minimum(exps, 1500.0 * len(kinds))) + 10 * n), (log, plain)


@pytest.mark.parametrize("bad", [math.nan, math.inf, -math.inf, 1e300, -1e300, 1e-320])
def test_products_with_odd_events(ctx, bad):
    """NaN, infinite, huge and subnormal columns give what the general form gives: the tile that
    holds one is evaluated by it, the others are untouched."""
    rng = np.random.default_rng(3)
    n = 5000
    for k, kinds in ((0, "GEX"), (1, "GEX"), (2, "GEX")):
        cols = [rng.uniform(-2.0, 2.0, n) for _ in range(3)]
        cols[k][[17, 4999]] = bad
        top = O.Prod("p", [_leaf(kind, OBS[j], j) for j, kind in enumerate(kinds)])
        ctx.set_program(*arrays(top)[1])
        ctx.upload_columns(cols)
        log, plain = _both(ctx)
        assert (math.isnan(log) and math.isnan(plain)) or log == plain or abs(log - plain) <= 1e-13 * abs(plain), \
            (k, log, plain)


def test_products_with_extreme_norms(ctx):
    """Norms outside 2^+-60, zero and negative: the general form for every tile."""
    rng = np.random.default_rng(4)
    top = O.Prod("p", [_leaf("G", OBS[0], 0), _leaf("E", OBS[1], 1)])
    f, p, c, o, nm = arrays(top)[1]
    ctx.set_program(f, p, c, o, nm)
    ctx.upload_columns([rng.uniform(-2.0, 2.0, 3000) for _ in range(2)])
    for scale in (1e-200, 1e200, 1e-310, 0.0, -1.0, math.nan):
        norms = np.array(nm, np.float64) * 1.0
        norms[-1] = scale
        ctx.update_norms(norms)
        log, plain = _both(ctx)
        assert (math.isnan(log) and math.isnan(plain)) or abs(log - plain) <= 1e-13 * abs(plain), (scale, log, plain)


def _gex(ctx, cols, width=0.7, resolution=0.4):
    top = O.Prod("p", [O.Gaussian("g", OBS[0], O.Var("m", 0.1), O.Var("s", width)), _leaf("E", OBS[1], 1),
                       O.ExpGaus("x", OBS[2], O.Var("xm", 0.0), O.Var("xs", resolution), O.Var("xr", 0.6))])
    ctx.set_program(*arrays(top)[1])
    ctx.upload_columns(cols)


def test_products_over_many_passes(ctx):
    """35 passes of the grid over the events, the last one ragged, with events outside the bound
    (a density of 0, a NaN, an infinite decay time) in single passes of some workgroups: the first,
    the 32nd and 33rd (two words of the bookkeeping), the last; one wave that meets them in so many
    passes that it stops trying.  A tile lost or added twice would move the sum by some 1000, the
    bound is 16 units of 2^-53 of the exponents' sum and of 10 an event."""
    cus, tile = 256, 1024  # one workgroup per CU, four events a lane
    n = 34 * cus * tile + 5 * tile + 77
    rng = np.random.default_rng(8)
    cols = [rng.uniform(-2.0, 2.0, n) for _ in range(3)]
    for block, passes in ((3, (31, 32)), (5, (0,)), (9, (32,)), (4, (1, 34)), (11, range(4, 34)), (6, range(34))):
        for k, t in enumerate(passes):
            e = (t * cus + block) * tile + 64 * (k % 4 if block != 11 else 1) + 256 * (k % 4) + k % 64
            cols[k % 3][e] = (100.0, math.nan, math.inf)[k % 3]
    cols[0][n - 1] = 100.0
    _gex(ctx, cols)
    try:
        ctx.set_tuning(capi.TUNE_BLOCKS_PER_CU, 1)
        log, plain = _both(ctx)
    finally:
        ctx.set_tuning(capi.TUNE_BLOCKS_PER_CU, 4)
    assert abs(log - plain) <= 16 * 2.0**-53 * 30 * n, (log, plain)


@pytest.mark.parametrize("n", [(1 << 20) - 1, (1 << 20) + 3])
def test_products_at_the_rule(ctx, n):
    """Either side of the size from which the logarithms are taken, by the default rule."""
    rng = np.random.default_rng(9)
    _gex(ctx, [rng.uniform(-2.0, 2.0, n) for _ in range(3)])
    auto = ctx.reduce_metric("NLL")[0]
    log, plain = _both(ctx)
    assert auto == (log if n >= 1 << 20 else plain)
    assert abs(log - plain) <= 16 * 2.0**-53 * 30 * n, (log, plain)


@pytest.mark.parametrize("case,bar", [("long decay times", 1.0), ("placeholders", 1.0), ("narrow", 1.35)])
@pytest.mark.parametrize("n", [1 << 20, 4_000_000])
def test_products_outside_the_bound_are_not_slow(ctx, case, bar, n):
    """Samples that meet the bound in most tiles: decay times to 330 widths of the resolution, and
    a tenth of the events at -999 (no reason to leave the logarithms: the factors are 2 and 0), and a
    width of 0.04 over +-2 (a twelfth of the events lies between the bound and a certain 0).  The bar
    is the time of the plain kernel's two-event form, which such samples leave behind by
    a fifth or, in the last, exceed by a fifth; a form that gives up whole tiles takes 1.45 times
    as long or more in each."""
    rng = np.random.default_rng(10)
    x, y = rng.uniform(-2.0, 2.0, n), rng.uniform(-2.0, 2.0, n)
    z = np.minimum(rng.exponential(1.5, n) + 0.03 * rng.standard_normal(n), 10.0)
    if case == "placeholders":
        x[rng.random(n) < 0.1] = -999.0
    _gex(ctx, [x, y, z], width=0.04 if case == "narrow" else 0.7,
         resolution=0.03 if case == "long decay times" else 0.4)
    us = {}
    try:
        for knob in (4, 2) * 3:
            ctx.set_tuning(capi.TUNE_FLAT, knob)
            us[knob] = min(us.get(knob, math.inf), 1e3 * ctx.time_sweep_back_to_back("NLL", 20))
    finally:
        ctx.set_tuning(capi.TUNE_FLAT, 1)
    log, plain = _both(ctx)
    assert abs(log - plain) <= 16 * 2.0**-53 * (3000 * n if case == "narrow" else 30 * n), (log, plain)
    assert us[4] <= bar * us[2], us
