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


@pytest.mark.parametrize("kinds", ["G", "X", "GEX", "XXGE", "GGEEXXGGEEXXGGEE", "GGEEXXGGEEXXGGEEX", "NG", "GZ", "U"])
@pytest.mark.parametrize("n", [1, 255, 1025, 70_001])
def test_products_in_logarithms(ctx, kinds, n):
    """One leaf, one to four columns, two leaves on a column, the most leaves the kernel takes
    and one more, densities that underflow in some tiles or are negative (those events add 0 in
    the reference's metric), from one event to a ragged end of the grid's second pass.  Every
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
    exps = sum(0.5 * (x / s) ** 2 if s else np.abs(x) + (1500 if "U" in kinds else 12) for x, s in
               ((cols[k % 4], {"G": 0.7, "N": 0.05}.get(kind)) for k, kind in enumerate(kinds)))
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
