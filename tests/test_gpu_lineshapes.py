"""Lineshapes of every kind, spin, channel, orientation and normalisation flag against the
oracle: the wave cache (all of it and single resonances), the grid integrals and the
time-dependent waves.

Tolerance: a wave is a product of a dozen correctly rounded factors, so engine and oracle
agree to some 1e-15 relative except where the pair's threshold factor 1 - (ma + mb)^2 / s
cancels, which multiplies the rounding by s / (s - (ma + mb)^2): below 1e3 on these samples."""
import time

import numpy as np
import pytest

import oracle as O
from goofit_amd import capi
from goofit_amd import workloads as W

pytestmark = pytest.mark.gpu

EQUAL = W.DALITZ_DECAY
UNEQUAL = (1.96834, 0.13957, 0.49368, 0.13498, 1.5, 5.0)  # three different daughters

SHAPES = {
    # kind, mass, width, spin, pair, norm
    "spins": [("RBW", 0.98, 0.06, s, p, True) for s in (0, 1, 2, 3) for p in (0, 1, 2)],
    "unnormalised": [("RBW", 0.9, 0.1, s, p, False) for s in (0, 1, 2) for p in (0, 1, 2)]
    + [("GS", 0.7758, 0.15, 1, 2, False)],
    "gs": [("GS", 0.7758, 0.15, s, p, True) for s in (0, 1, 2) for p in (0, 1, 2)] + [("NONRES", 0, 0, 0, 0, True)],
    "symmetrised": [("SYM", 0.9, 0.1, s, p, n) for s in (0, 1, 2) for p in (0, 2) for n in (True, False)],
    "one": [("NONRES", 0, 0, 0, 0, True)],
    # a plan's terms in the kernels' arguments, 16 of them, and one more
    "args": [("RBW", 0.7 + 0.05 * k, 0.1, k % 3, k % 3, True) for k in range(14)] + [("SYM", 0.9, 0.1, 1, 0, True)],
    "args and one": [("GS", 0.7758, 0.15, 1, 2, True)] + [("RBW", 0.7 + 0.05 * k, 0.1, k % 3, k % 3, True) for k in range(14)]
    + [("SYM", 0.9, 0.1, 1, 0, True)],
}


def _model(shapes, decay, td=False):
    m12, m13 = O.Obs("m12", 0.0, 3.5, 60), O.Obs("m13", 0.0, 3.5, 60)
    num = O.Obs("evt", 0.0, 1e9, 1, event_number=True)
    res = []
    for k, (kind, mass, width, spin, pair, norm) in enumerate(shapes):
        a = (O.Var(f"re{k}", 0.3 + 0.1 * k), O.Var(f"im{k}", 0.7 - 0.2 * k))
        mw = (O.Var(f"m{k}", mass), O.Var(f"w{k}", width))
        if kind == "NONRES":
            res.append(O.NonRes(f"r{k}", *a))
        elif kind == "GS":
            res.append(O.GS(f"r{k}", *a, *mw, spin, pair, norm))
        else:
            res.append(O.RBW(f"r{k}", *a, *mw, spin, pair, norm, sym=kind == "SYM"))
    eff = O.MultiPolynomial("eff", [m12, m13], [O.Var("one", 1.0)], [O.Var("z0", 0.0), O.Var("z1", 0.0)], 0)
    if td:
        t, s = O.Obs("t", -2.0, 20.0), O.Obs("s", 0.0, 0.8)
        mix = [O.Var(n, v) for n, v in zip(("tau", "x", "y", "dx", "dy"), W.TD_MIX)]
        return O.Tddp("td", t, s, m12, m13, num, decay, mix, res, O.TruthResolution(), eff), res
    return O.Dalitz("dalitz", m12, m13, num, decay, res, eff), res


def _events(n, decay, seed):
    m12, m13 = W.dalitz_uniform(n, seed, decay)
    rng = np.random.default_rng(seed)
    out = rng.choice(n, n // 10, replace=False)  # a tenth outside the plot
    m12[out], m13[out] = rng.uniform(0.0, 3.5, (2, out.size))
    return m12, m13


def _close(got, ref):
    np.testing.assert_allclose(got, ref, rtol=1e-12, atol=1e-13 * np.abs(ref).max())


@pytest.mark.parametrize("decay", [EQUAL, UNEQUAL], ids=["equal", "unequal"])
@pytest.mark.parametrize("shapes", sorted(SHAPES))
def test_waves_and_integrals(ctx, shapes, decay):
    top, res = _model(SHAPES[shapes], decay)
    for n in (1, 63, 257, 3001):  # ragged waves and workgroups
        m12, m13 = _events(n, decay, 17 + n)
        if n == 1:
            m12, m13 = np.array([1.0]), np.array([1.0])
        aos = np.stack([m12, m13, np.arange(n, dtype=np.float64)], 1)
        M = O.Model(top, aos, decay=decay)
        M.op.sync_params()
        ctx.set_program(*M.op.prog.arrays())
        ctx.set_decay(decay)
        ctx.upload_columns([m12, m13, aos[:, 2]])
        ctx.set_identity_column(2)
        ctx.dalitz_set_data_size(0, n)
        ctx.dalitz_cache(0)
        funcs, eff = M.op.dalitz_layout(0)
        inside = W.in_dalitz_np(m12, m13, decay)
        for i, f in enumerate(funcs):
            got = ctx.dalitz_get_cache(0, i, n)
            assert np.all(got[~inside] == 0)
            if inside.any():
                _close(got, M.op.dalitz_wave(0, f, aos))
    # one resonance at a time: the others keep their values
    before = [ctx.dalitz_get_cache(0, i, n) for i in range(len(funcs))]
    for i in {0, len(funcs) - 1}:
        if SHAPES[shapes][i][0] == "NONRES":
            continue
        p = M.op.p.copy()
        at = top.components[i].parameters_idx + 1
        p[at] *= 1.01
        ctx.update_params(p)
        ctx.dalitz_cache(0, 1 << i)
        for k in range(len(funcs)):
            same = np.array_equal(ctx.dalitz_get_cache(0, k, n), before[k])
            assert same == (k != i)
        ctx.update_params(M.op.p)
        ctx.dalitz_cache(0, 1 << i)
        assert np.array_equal(ctx.dalitz_get_cache(0, i, n), before[i])
    for nb in (1, 8, 61):  # fewer cells than a wave; none inside; ragged
        grid6 = [0.0, 3.5, nb, 0.0, 3.5, nb]
        ref = M.op.dalitz_integrals(0, grid6, eff)
        got = ctx.dalitz_gram(0, grid6, eff, len(funcs))
        np.testing.assert_allclose(got, ref, rtol=1e-11, atol=1e-12 * max(np.abs(ref).max(), 1e-300))


@pytest.mark.parametrize("shapes", ["gs", "symmetrised"])
@pytest.mark.parametrize("nb", [362, 363, 401])
def test_integrals_over_more_cells_than_a_pass(ctx, shapes, nb):
    """A pass of the integral's grid takes 512 workgroups x 256 cells = 131072: one pass and all but
    28 cells of it (362^2), 697 cells of a second (363^2), and a fifth of one more, so that waves take
    their LDS rows again, some of them for a tile with no cell inside the plot."""
    top, res = _model(SHAPES[shapes], UNEQUAL)
    M = O.Model(top, np.zeros((1, 3)), decay=UNEQUAL)
    M.op.sync_params()
    ctx.set_program(*M.op.prog.arrays())
    ctx.set_decay(UNEQUAL)
    funcs, eff = M.op.dalitz_layout(0)
    grid6 = [0.0, 3.5, nb, 0.0, 3.5, nb]
    ref = M.op.dalitz_integrals(0, grid6, eff)
    np.testing.assert_allclose(ctx.dalitz_gram(0, grid6, eff, len(funcs)), ref, rtol=1e-11,
                               atol=1e-12 * np.abs(ref).max())


@pytest.mark.parametrize("shapes", ["spins", "gs", "symmetrised"])
def test_time_dependent_waves(ctx, shapes):
    """The B waves: every lineshape at the reversed point (a pair below its threshold there).  Alone,
    a resonance's terms are in the kernel's arguments, with the others on the device: the same
    bits."""
    n, decay = 1000, UNEQUAL
    top, res = _model(SHAPES[shapes], decay, td=True)
    m12, m13 = _events(n, decay, 5)
    aos = np.stack([np.full(n, 0.5), np.full(n, 0.05), m12, m13, np.arange(n, dtype=np.float64)], 1)
    M = O.Model(top, aos, decay=decay)
    M.op.sync_params()
    ctx.set_program(*M.op.prog.arrays())
    ctx.set_decay(decay)
    ctx.upload_columns(list(aos.T.copy()))
    ctx.set_identity_column(4)
    ctx.dalitz_set_data_size(0, n)
    ctx.dalitz_cache(0)
    funcs = M.op.tddp_layout(0)[0]
    for i, f in enumerate(funcs):
        a, b = M.op.tddp_wave(0, f, aos)
        _close(ctx.dalitz_get_cache(0, i, n), a)
        _close(ctx.dalitz_get_cache(0, len(funcs) + i, n), b)
    before = [ctx.dalitz_get_cache(0, i, n) for i in range(2 * len(funcs))]
    ctx.dalitz_set_data_size(0, n)
    for i in range(len(funcs)):
        ctx.dalitz_cache(0, 1 << i)
    for i, w in enumerate(before):
        assert np.array_equal(ctx.dalitz_get_cache(0, i, n), w)


def _mix64(z):
    """The finaliser of the counter-based stream (splitmix64)."""
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _unif(key, counter):
    return (_mix64(key ^ _mix64(counter)) >> np.uint64(11)) * 2.0 ** -53


def _stream(ctx, shapes, box, seed, passes, decay=EQUAL):
    """The documented stream's candidates over the given passes of 2^22: their points, their
    uniform numbers, and the values (0 outside the plot), and a program that generates from it."""
    top, res = _model(shapes, decay)
    with np.errstate(over="ignore"):
        key = _mix64(np.array([seed], np.uint64) ^ np.uint64(0x6A09E667F3BCC909))[0]
        i = np.arange(passes << 22, dtype=np.uint64)
        m12 = box[0] + _unif(key, np.uint64(2) * i) * (box[1] - box[0])
        m13 = box[2] + _unif(key, np.uint64(2) * i + np.uint64(1)) * (box[3] - box[2])
        u = _unif(key ^ np.uint64(0xD1B54A32D192ED03), i)
    inside = np.nonzero(W.in_dalitz_np(m12, m13, decay))[0]
    M = O.Model(top, np.zeros((1, 3)), decay=decay)
    M.op.sync_params()
    ctx.set_program(*M.op.prog.arrays())
    ctx.set_decay(decay)
    ctx.upload_columns([m12[inside], m13[inside], np.arange(inside.size, dtype=np.float64)])
    ctx.set_identity_column(2)
    ctx.dalitz_set_data_size(0, inside.size)
    ctx.dalitz_cache(0)
    return m12, m13, u, inside, ctx.eval_metric("EVAL")


SHORT = [("RBW", 0.7758, 0.15, 1, 0, True), ("NONRES", 0, 0, 0, 0, True), ("GS", 0.7758, 0.15, 1, 2, True),
         ("SYM", 0.98, 0.06, 0, 1, True)]
LONG = SHORT + [("SYM", 0.8 + 0.05 * k, 0.1, k % 3, k % 3, True) for k in range(7)]  # 19 terms: the plan on the device


@pytest.mark.parametrize("shapes,fmax", [(SHORT, 4000.0), (LONG, None)], ids=["short", "long"])
def test_generated_events_are_the_stream(ctx, shapes, fmax):
    """The accepted candidates of the documented stream, in its order, over one pass of 2^22
    and into the second; a few events, a whole pass, one more than a pass; a box that cuts
    the plot and one that misses it."""
    seed, box = 23, [0.2, 2.6, 0.1, 3.0]
    m12, m13, u, inside, value = _stream(ctx, shapes, box, seed, 2)
    fmax = fmax or 1.01 * value.max()
    assert value.max() < fmax
    keep = inside[u[inside] * fmax < value]
    first = int(np.sum(keep < 1 << 22))
    assert 1000 < first < keep.size
    for n in (1, 777, first, first + 1, keep.size):
        a, b, tried, top_value = ctx.dalitz_generate(0, n, seed, box, fmax)
        assert np.array_equal(a, m12[keep[:n]]) and np.array_equal(b, m13[keep[:n]])
        assert tried == (1 if n <= first else 2) << 22 and top_value == fmax
    # the envelope found from the first pass, whose candidates are then not used again
    n = keep.size - first
    a, b, tried, top_value = ctx.dalitz_generate(0, n // 2, seed, box)
    top_seen = value[inside < 1 << 22].max()
    np.testing.assert_allclose(top_value, 1.25 * top_seen, rtol=1e-13)
    later = inside[(inside >= 1 << 22) & (u[inside] * top_value < value)]
    k = min(later.size, n // 2)
    assert np.array_equal(a[:k], m12[later[:k]]) and np.array_equal(b[:k], m13[later[:k]])
    # an envelope below the values, and a box without the plot
    with pytest.raises(capi.GooFitError, match="raise fmax"):
        ctx.dalitz_generate(0, 10, seed, box, 0.5 * top_seen)
    with pytest.raises(capi.GooFitError, match="is zero"):
        ctx.dalitz_generate(0, 10, seed, [2.95, 3.0, 2.95, 3.0])
    a2, b2, _, _ = ctx.dalitz_generate(0, 777, seed, box, fmax)
    assert np.array_equal(a2, m12[keep[:777]]) and np.array_equal(b2, m13[keep[:777]])


def test_generated_events_of_queued_passes(ctx):
    """A low acceptance, which needs six passes: one alone, then the others queued together, as
    many as the first one's acceptance asks for.  Counts just below and just above a pass's
    end, where one pass too many is queued, which finds the rows complete and must leave them."""
    seed, box, passes = 31, [0.0, 3.0, 0.0, 3.0], 6
    m12, m13, u, inside, value = _stream(ctx, SHORT, box, seed, passes)
    fmax = 40.0 * value.max()
    keep = inside[u[inside] * fmax < value]
    ends = np.searchsorted(keep, np.arange(1, passes + 1) << 22)
    assert ends[0] > 1000 and np.all(np.diff(ends) > 1000)
    ahead = 0
    for end in ends[1:5]:
        for n in (end - 1, end, end + 1):
            a, b, tried, top_value = ctx.dalitz_generate(0, int(n), seed, box, fmax)
            assert np.array_equal(a, m12[keep[:n]]) and np.array_equal(b, m13[keep[:n]])
            need = int(np.searchsorted(ends, n)) + 1
            assert tried == need << 22 and top_value == fmax
            ahead += 1 + int(np.ceil((n - ends[0]) / ends[0])) > need
    assert ahead  # at least one of the calls queued a pass that it did not need


def test_refresh_of_one_resonance_is_not_slow(ctx):
    """One resonance of sixteen over a small sample is the work of a model's only one: what is
    prepared for a call must not grow with the others (a sixth more with all of their constants
    formed on the device in front of it)."""
    us = {}
    for nres in (1, 16) * 3:
        top, _ = _model([("RBW", 0.7 + 0.05 * k, 0.1, k % 3, k % 3, True) for k in range(nres)], EQUAL)
        n = 1000
        m12, m13 = _events(n, EQUAL, 3)
        M = O.Model(top, np.zeros((1, 3)), decay=EQUAL)
        M.op.sync_params()
        ctx.set_program(*M.op.prog.arrays())
        ctx.set_decay(EQUAL)
        ctx.upload_columns([m12, m13, np.arange(n, dtype=np.float64)])
        ctx.set_identity_column(2)
        ctx.dalitz_set_data_size(0, n)
        t = []
        for _ in range(200):
            a = time.perf_counter()
            ctx.dalitz_cache(0, 1)
            t.append(time.perf_counter() - a)
        us[nres] = min(us.get(nres, np.inf), 1e6 * np.median(t))
    assert us[16] <= 1.1 * us[1], us
