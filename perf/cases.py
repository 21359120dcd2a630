"""The work that users of the likelihood engine have it do, as measurable cases.

Each case goes through a public entry point: the C ABI of include/goofit_hip.h (module
goofit_amd.capi, one context per state) for the calls that a minimiser makes thousands of
times, and the GooFit API (UnbinnedDataSet, FitManager, BatchFitter) for whole fits.  The
models and sizes are those of goofit_amd/workloads.py, of bench.py and of the tests.

`exact` states the same results in 64-bit torch from the formulas alone.
"""
import math

import numpy as np
import torch

from goofit_amd import capi
from goofit_amd import workloads as W

F64 = torch.float64
DEV = "cuda"

# --------------------------------------------------------------------------- cases


def listed():
    return [
        # one likelihood call of a 1-D signal + background fit on a toy-sized sample: the
        # smallest call there is, launch and read-back latency
        dict(name="add1d_nll_10k", kind="add1d", n=10_000),
        # one likelihood call of an unbinned 3-D fit on a large sample (bench.py's prod3d)
        dict(name="prod3d_nll_10m", kind="prod3d", n=10_000_000),
        # one likelihood call of a two-dimensional mass x decay-time fit, signal and background
        # each a product, with two shapes that are normalised on a grid at every call
        dict(name="mixture_nll_1m", kind="mixture", n=1_000_003, degree=2, nbins=2000),
        # the headline: one likelihood call of the 16-resonance Dalitz fit on 1e6 events
        dict(name="dalitz16_nll_1m", kind="dalitz_nll", n=1_000_000, nres=16),
        # the same call on a sample of a typical toy's size and a smaller model
        dict(name="dalitz6_nll_50k", kind="dalitz_nll", n=50_021, nres=6),
        # the derivative round that MIGRAD asks for: two points for each of 30 couplings
        dict(name="dalitz16_round_1m", kind="dalitz_round", n=1_000_000, nres=16, sets=60),
        # what a changed mass or width costs: every lineshape over the events, the
        # normalisation integrals on the grid, and the events' likelihood values
        dict(name="dalitz16_lineshapes_1m", kind="lineshapes", n=1_000_000, nres=16, grid=1414),
        # one likelihood call of a time-dependent fit: three-Gaussian resolution, mistag, tag
        dict(name="tddp16_nll_1m", kind="tddp", n=1_000_000, nres=16, threegauss=True, mistag=True),
        # toy generation from the 16-resonance model by accept-reject
        dict(name="dalitz16_generate_200k", kind="generate", n=200_000, nres=16),
        # a whole Dalitz fit through the GooFit API: data in, caches, MIGRAD, errors
        dict(name="dalitz16_fit_200k", kind="fit", n=200_000, nres=16, grid=500),
        # a batch of toy fits of the 8-resonance model
        dict(name="dalitz8_toys_64", kind="toys", toys=64, n=30_000, nres=8, grid=400),
        # training of the importance-sampling proposal of the normalisation integral
        dict(name="proposal_train_8k", kind="train", n=500_000, steps=40, batch=8192),
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["add1d", "prod3d", "mixture", "dalitz_nll", "dalitz_round", "lineshapes", "tddp", "generate",
                       "fit", "toys", "train"])
    if kind == "add1d":
        return dict(kind=kind, n=_log(rng, 3_000, 1_000_000))
    if kind == "prod3d":
        return dict(kind=kind, n=_log(rng, 50_000, 10_000_000))
    if kind == "mixture":
        return dict(kind=kind, n=_log(rng, 20_000, 2_000_000), degree=rng.randint(1, 4),
                    nbins=rng.choice([500, 1000, 2000]))
    nres = rng.randint(3, 16)
    if kind == "dalitz_nll":
        return dict(kind=kind, n=_log(rng, 5_000, 1_500_000), nres=nres)
    if kind == "dalitz_round":
        return dict(kind=kind, n=_log(rng, 20_000, 1_000_000), nres=nres, sets=rng.randint(2, 2 * (2 * nres - 2)))
    if kind == "lineshapes":
        return dict(kind=kind, n=_log(rng, 20_000, 1_000_000), nres=nres, grid=rng.randint(150, 1500))
    if kind == "tddp":
        return dict(kind=kind, n=_log(rng, 20_000, 1_000_000), nres=nres, threegauss=rng.random() < 0.6,
                    mistag=rng.random() < 0.5)
    if kind == "generate":
        return dict(kind=kind, n=_log(rng, 5_000, 200_000), nres=nres)
    if kind == "fit":
        return dict(kind=kind, n=_log(rng, 50_000, 200_000), nres=rng.randint(5, 16), grid=rng.randint(200, 500))
    if kind == "toys":
        return dict(kind=kind, toys=rng.randint(8, 64), n=_log(rng, 10_000, 30_000), nres=rng.randint(4, 8), grid=400)
    return dict(kind=kind, n=_log(rng, 50_000, 500_000), steps=rng.randint(10, 40),
                batch=128 * rng.randint(8, 64))


# ------------------------------------------------------------------- Dalitz formulas

DECAY = W.DALITZ_DECAY
MOTHER, D1, D2, D3, R_MESON, R_MOTHER = DECAY
BOX = (0.0, 3.0, 0.0, 3.0)  # m12 and m13 of the models' observables
PI = 3.14159265359          # as the Gounaris-Sakurai form of the reference has it
CHUNK = 1 << 21


def _table(nres):
    """The first nres resonances of the 16-resonance model."""
    return W.DALITZ_RESONANCES[:nres]


def _couplings(nres):
    return W.dalitz_couplings(3, nres)


def _breakup(s, a, b):
    """sqrt(1 - (a + b)^2 / s) sqrt(1 - (a - b)^2 / s), a factor below its threshold taken as 1."""
    out = 1.0
    for m in (a + b, a - b):
        k = 1 - m * m / s
        out = out * torch.where(k >= 0, torch.sqrt(k.clamp(min=0)), torch.ones_like(k))
    return out


def _cm_momentum(s, a, b):
    s = torch.as_tensor(s, dtype=F64)
    return 0.5 * torch.sqrt(s) * _breakup(s, a, b)


def _mother_momentum(s, mother, bachelor):
    s = torch.as_tensor(s, dtype=F64)
    return 0.5 * s * _breakup(s, mother, bachelor) / mother


def _inside(m12, m13):
    m23 = MOTHER ** 2 + D1 ** 2 + D2 ** 2 + D3 ** 2 - m12 - m13
    s = torch.sqrt(m12)
    e1 = 0.5 * (m12 - D2 * D2 + D1 * D1) / s
    e3 = 0.5 * (MOTHER * MOTHER - m12 - D3 * D3) / s
    p1, p3 = torch.sqrt(e1 * e1 - D1 * D1), torch.sqrt(e3 * e3 - D3 * D3)
    lo, hi = (e1 + e3) ** 2 - (p1 + p3) ** 2, (e1 + e3) ** 2 - (p1 - p3) ** 2
    ok = (m23 >= 0) & (m23 <= (MOTHER - D1) ** 2) & (m12 >= (D1 + D2) ** 2) & (m12 <= (MOTHER - D3) ** 2)
    return ok & ~(m13 < lo) & ~(m13 > hi)


def _wave(entry, m12, m13, m23):
    """(re, im) of one resonance at points inside the Dalitz plot."""
    _, kind, mass, width, spin, pair = entry
    if kind == "NONRES":
        return torch.ones_like(m12), torch.zeros_like(m12)
    s = (m12, m13, m23)[pair]
    da, db = (D1 if pair != 2 else D2), (D2 if pair == 0 else D3)
    bachelor = (D3, D2, D1)[pair]
    m2 = mass * mass
    q, q0 = _cm_momentum(s, da, db), float(_cm_momentum(m2, da, db))
    p, p0 = _mother_momentum(s, MOTHER, bachelor), float(_mother_momentum(m2, MOTHER, bachelor))
    barrier, barrier_mother = torch.ones_like(s), torch.ones_like(s)
    if spin:
        def form(k, r):
            z = (r * k) ** 2
            return 1 + z if spin == 1 else 9 + 3 * z + z * z
        barrier = form(q0, R_MESON) / form(q, R_MESON)
        barrier_mother = form(p0, R_MOTHER) / form(p, R_MOTHER)
    running = (q / q0) ** (2 * spin + 1) * barrier
    if kind == "GS":
        a, b = D2, D3

        def h(t):
            k, r = _cm_momentum(t, a, b), torch.sqrt(torch.as_tensor(t, dtype=F64))
            return 2 / PI * (k / r) * torch.log((r + 2 * k) / (a + b))

        k, k0 = _cm_momentum(s, a, b), _cm_momentum(m2, a, b)
        dh = h(m2) * (1 / (8 * k0 * k0) - 1 / (2 * m2)) + 1 / (2 * PI * m2)
        f = width * m2 / k0 ** 3 * (k * k * (h(s) - h(m2)) + (m2 - s) * k0 * k0 * dh)
        sm24 = (a + b) ** 2 / 4
        d = (3 / PI * sm24 / (k0 * k0) * torch.log((mass + 2 * k0) / (a + b)) + mass / (2 * PI * k0)
             - sm24 * mass / (PI * k0 ** 3))
        top = 1 + d * width / mass
        u, v = m2 - s + f, mass * width * running
        re, im = top * u / (u * u + v * v), top * v / (u * u + v * v)
    else:
        u, v = m2 - s, m2 * width * running / torch.sqrt(s)
        re, im = u / (u * u + v * v), v / (u * u + v * v)
    scale = torch.sqrt(barrier * barrier_mother)
    if spin:
        ma, mb, mc = ((D1, D2, D3), (D3, D1, D2), (D2, D3, D1))[pair]
        sac, sbc, sab = ((m13, m23, m12), (m23, m12, m13), (m12, m13, m23))[pair]
        zemach = -((sbc - sac) + (MOTHER ** 2 - mc ** 2) * (ma ** 2 - mb ** 2) / sab)
        if spin == 2:
            one = sab - 2 * MOTHER ** 2 - 2 * mc ** 2 + (MOTHER ** 2 - mc ** 2) ** 2 / sab
            two = sab - 2 * ma ** 2 - 2 * mb ** 2 + (ma ** 2 - mb ** 2) ** 2 / sab
            zemach = zemach ** 2 - one * two / 3
        scale = scale * zemach
    return re * scale, im * scale


def _waves(nres, m12, m13, swap=False):
    """[nres, n] complex waves, 0 outside the plot (swap: at the point (m13, m12))."""
    m23 = MOTHER ** 2 + D1 ** 2 + D2 ** 2 + D3 ** 2 - m12 - m13
    ok = _inside(m12, m13)
    a, b = (m13, m12) if swap else (m12, m13)
    out = torch.empty(nres, m12.numel(), dtype=torch.complex128, device=m12.device)
    for i, entry in enumerate(_table(nres)):
        re, im = _wave(entry, a, b, m23)
        out[i] = torch.where(ok, torch.complex(re, im), torch.zeros((), dtype=torch.complex128, device=m12.device))
    return out


def _amplitude(nres, c, m12, m13, swap=False):
    """sum_i c_i W_i, in pieces."""
    c = torch.as_tensor(np.asarray(c, np.complex128), device=m12.device)
    return torch.cat([(c[:, None] * _waves(nres, x, y, swap)).sum(0)
                      for x, y in zip(m12.split(CHUNK), m13.split(CHUNK))])


def _cells(grid):
    """Centres of the integration cells that lie in the Dalitz plot, and the area of one."""
    x = (torch.arange(grid, dtype=F64, device=DEV) + 0.5) * (3.0 / grid)
    m12, m13 = x.repeat(grid), x.repeat_interleave(grid)
    ok = _inside(m12, m13)
    return m12[ok], m13[ok], (3.0 / grid) ** 2


def _integrals(nres, grid):
    """sum over the cells of B_i conj(B_j)."""
    m12, m13, _ = _cells(grid)
    out = torch.zeros(nres, nres, dtype=torch.complex128, device=DEV)
    for x, y in zip(m12.split(CHUNK), m13.split(CHUNK)):
        w = _waves(nres, x, y)
        out += w @ w.conj().T.contiguous()
    return out


_kept = {}  # integrals and envelopes by (nres, grid): the same for every seed


def _norm(nres, c, grid):
    """1 / integral of |sum c_i B_i|^2 over the plot."""
    key = (nres, grid)
    if key not in _kept:
        _kept[key] = _integrals(nres, grid).cpu().numpy()
    c = np.asarray(c, np.complex128)
    return float(1.0 / ((c[:, None] * c.conj()[None, :] * _kept[key]).sum().real * (3.0 / grid) ** 2))


def _dalitz_events(n, nres, seed):
    """n events of the model by accept-reject on uniform points, on the GPU."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    c = _couplings(nres)
    key = ("top", nres)
    if key not in _kept:
        m12, m13, _ = _cells(1000)
        _kept[key] = float(_amplitude(nres, c, m12, m13).abs().square().max()) * 1.2
    got, have = [], 0
    while have < n:
        m12, m13 = (torch.rand(2, 1 << 22, dtype=F64, device=DEV, generator=gen) * 3.0).unbind(0)
        ok = _inside(m12, m13)
        m12, m13 = m12[ok], m13[ok]
        v = _amplitude(nres, c, m12, m13).abs().square()
        take = torch.rand(v.numel(), dtype=F64, device=DEV, generator=gen) * _kept[key] < v
        got.append(torch.stack([m12[take], m13[take]]))
        have += got[-1].shape[1]
    m12, m13 = torch.cat(got, 1)[:, :n]
    return m12.contiguous(), m13.contiguous()


# ------------------------------------------------------------------ flattened models
#
# A node is (function, parameters, constants, observable indices, children); the arrays are
# the flattened tree of include/goofit_hip.h.


def _flatten(node):
    funcs, params, consts, obs, norms = [], [], [], [], []

    def put(f, p, c, o, kids):
        funcs.append(f)
        params.extend([len(p), *p])
        consts.extend([len(c), *c])
        obs.extend([len(o), *o])
        norms.extend([1.0, 1.0])
        for k in kids:
            put(*k)

    put(*node)
    return (np.asarray(funcs, np.int32), *(np.asarray(a, np.float64) for a in (params, consts, obs, norms)))


def _dalitz_node(nres, c):
    eff = (capi.FN["MULTI_POLYNOMIAL"], [0.0, 0.0, 1.0], [0.0, 1.0, 2.0], [0, 1], [])
    kids = [(capi.FN["NONRES"], [], [], [], []) if kind == "NONRES" else
            (capi.FN["GS" if kind == "GS" else "RBW"], [mass, width], [spin, pair, 1.0], [], [])
            for _, kind, mass, width, spin, pair in _table(nres)]
    return (capi.FN["DALITZ"], np.column_stack([c.real, c.imag]).ravel().tolist(), [nres, 0.0], [0, 1, 2], kids + [eff])


def _dalitz_context(nres, m12, m13):
    ctx = capi.Context(0)
    arrays = _flatten(_dalitz_node(nres, _couplings(nres)))
    ctx.set_program(*arrays)
    ctx.set_decay(DECAY)
    n = m12.numel()
    ctx.upload_columns([m12.cpu().numpy(), m13.cpu().numpy(), np.arange(n, dtype=np.float64)])
    ctx.set_identity_column(2)
    ctx.dalitz_set_data_size(0, n)
    return ctx, arrays


def _with_couplings(params, c):
    p = params.copy()
    p[1:1 + 2 * len(c)] = np.column_stack([c.real, c.imag]).ravel()
    return p


def _moved(nres, seed):
    """The couplings of a likelihood call: the model's, a few per cent off."""
    r = np.random.default_rng(seed + 77)
    c = _couplings(nres)
    return c * (1 + 0.03 * r.standard_normal(nres)) * np.exp(0.03j * r.standard_normal(nres))


def _round_sets(case, seed):
    """A derivative round: the base point with one real parameter up or down per set."""
    base = _moved(case["nres"], seed)
    sets = []
    for k in range(case["sets"]):
        c = base.copy()
        j = (k // 2) % (2 * len(c))
        step = (1e-3 if k % 2 == 0 else -1e-3) * (1.0 if j % 2 == 0 else 1j)
        c[j // 2] += step
        sets.append(c)
    return sets


def _truncated(gen, n, draw_some, lo, hi):
    got, have = [], 0
    while have < n:
        x = draw_some(max(2 * (n - have), 1024), gen)
        x = x[(x >= lo) & (x <= hi)]
        got.append(x)
        have += x.numel()
    return torch.cat(got)[:n]


def _gauss(gen, n, mu, sigma, lo, hi):
    return _truncated(gen, n, lambda k, g: mu + sigma * torch.randn(k, dtype=F64, device=DEV, generator=g), lo, hi)


def _expo(gen, n, alpha, lo, hi):
    u = torch.rand(n, dtype=F64, device=DEV, generator=gen)
    return torch.log(math.exp(alpha * lo) + u * (math.exp(alpha * hi) - math.exp(alpha * lo))) / alpha


def _decay_time(gen, n, sigma, tau, lo, hi):
    def some(k, g):
        e = -tau * torch.log1p(-torch.rand(k, dtype=F64, device=DEV, generator=g))
        return e + sigma * torch.randn(k, dtype=F64, device=DEV, generator=g)
    return _truncated(gen, n, some, lo, hi)


def _shape_params(case, seed):
    """Parameter values of a likelihood call of the 1-D, 3-D and 2-D models."""
    r = np.random.default_rng(seed + 5)

    def near(v):
        return float(v * (1 + 0.02 * r.standard_normal()))
    if case["kind"] == "add1d":
        return dict(mu=near(0.3), sigma=near(0.8), alpha=near(-0.4), frac=near(0.3))
    if case["kind"] == "prod3d":
        return dict(mu=0.01 * float(r.standard_normal()), sigma=near(1.0), alpha=near(-1.2), rate=near(1 / 1.5))
    return dict(frac=near(0.4), mu=near(0.2), sigma=near(0.5), rate=near(1 / 1.5), slope=near(-0.9),
                poly=[near(1.0)] + [near(0.25 / (k * k)) for k in range(1, case["degree"] + 1)])


def _shape_columns(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    n = case["n"]
    if case["kind"] == "add1d":
        sig = int(0.3 * n)
        x = torch.cat([_gauss(gen, sig, 0.3, 0.8, -5, 5), _expo(gen, n - sig, -0.4, -5, 5)])
        return [x[torch.randperm(n, device=DEV, generator=gen)]]
    if case["kind"] == "prod3d":
        return [_gauss(gen, n, 0.0, 1.0, -6, 6), _expo(gen, n, -1.2, 0, 8), _decay_time(gen, n, 0.1, 1.5, 0, 10)]
    sig = int(0.4 * n)
    u = torch.rand(n - sig, dtype=F64, device=DEV, generator=gen)
    x = torch.cat([_gauss(gen, sig, 0.2, 0.5, -3, 3), 6 * u - 3])
    t = torch.cat([_decay_time(gen, sig, 0.1, 1.5, 0, 10), _expo(gen, n - sig, -0.9, 0, 10)])
    order = torch.randperm(n, device=DEV, generator=gen)
    return [x[order], t[order]]


def _shape_node(case, v):
    F = capi.FN
    if case["kind"] == "add1d":
        return (F["ADD"], [v["frac"]], [], [0], [(F["GAUSSIAN"], [v["mu"], v["sigma"]], [], [0], []),
                                                 (F["EXP"], [v["alpha"]], [], [0], [])])
    if case["kind"] == "prod3d":
        return (F["PROD"], [], [3], [0, 1, 2], [(F["GAUSSIAN"], [v["mu"], v["sigma"]], [], [0], []),
                                                (F["EXP"], [v["alpha"]], [], [1], []),
                                                (F["EXPGAUS"], [0.0, 0.1, v["rate"]], [], [2], [])])
    signal = (F["PROD"], [], [2], [0, 1], [(F["GAUSSIAN"], [v["mu"], v["sigma"]], [], [0], []),
                                           (F["EXPGAUS"], [0.0, 0.1, v["rate"]], [], [1], [])])
    background = (F["PROD"], [], [2], [0, 1], [(F["POLYNOMIAL"], v["poly"], [0.0], [0], []),
                                               (F["EXP"], [v["slope"]], [], [1], [])])
    return (F["ADD"], [v["frac"]], [], [0, 1], [signal, background])


def _exp_integral(a, lo, hi):
    return (math.exp(a * hi) - math.exp(a * lo)) / a


def _expgaus(x, mean, sigma, alpha):
    arg = (mean + alpha * sigma * sigma - x) / (sigma * 1.4142135623)
    return 0.5 * alpha * torch.exp(0.5 * alpha * (2 * mean + alpha * sigma * sigma - 2 * x)) * torch.erfc(arg)


def _grid1(lo, hi, nbins):
    return ((hi - lo) / nbins) * (torch.arange(nbins, dtype=F64, device=DEV) + 0.5) + lo


TG = (0.7, 0.2, 0.05, 1.1, -0.1, 2.0, 0.0, 6.0, 0.0, 0.01, 1.05, 0.0, 1.0)  # three-Gaussian resolution
MIX = W.TD_MIX


def _td_columns(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    n = case["n"]
    m12, m13 = _dalitz_events(n, case["nres"], seed)
    t = -MIX[0] * torch.log1p(-torch.rand(n, dtype=F64, device=DEV, generator=gen))
    s = 0.03 + 0.05 * torch.rand(n, dtype=F64, device=DEV, generator=gen)
    cols = [t, s, m12, m13, torch.arange(n, dtype=F64, device=DEV)]
    if case["mistag"]:
        cols.append(0.3 * torch.rand(n, dtype=F64, device=DEV, generator=gen))
        cols.append(2.0 * torch.randint(0, 2, (n,), device=DEV, generator=gen).to(F64) - 1.0)
    return cols


def _td_mix(seed):
    r = np.random.default_rng(seed + 9)
    return [MIX[0] * (1 + 0.01 * float(r.standard_normal())), MIX[1], MIX[2], 0.0, 0.0]


def _td_node(case, mix):
    c = _couplings(case["nres"])
    top = _dalitz_node(case["nres"], c)
    res = (20, list(TG), [], [], []) if case["threegauss"] else (19, [], [], [], [])  # GF_FN_*_RES
    kids = top[4][:-1] + [res, (top[4][-1][0], top[4][-1][1], top[4][-1][2], [2, 3], [])]
    obs = [0, 1, 2, 3, 4] + ([5, 6] if case["mistag"] else [])
    end = 1 + len(kids)
    return (18, [*mix, *top[1]], [case["nres"], 0.0, 0.0 if case["mistag"] else 1.0, float(end)], obs, kids)  # GF_FN_TDDP


def _td_norm(case):
    """The size of the time-dependent model's integral (mixing left out)."""
    return _norm(case["nres"], _couplings(case["nres"]), 300) / (2 * MIX[0])


TRAIN_LR, TRAIN_SEED = 6e-3, 11


def _net_params(seed):
    """Initial weights of the proposal network: W1[128][2], b1, W2[128][128], b2, w3, b3."""
    r = np.random.default_rng(seed + 13)
    b2 = math.sqrt(6 / 128)
    return np.concatenate([r.uniform(-3, 3, 384), r.uniform(-b2, b2, 128 * 128), np.zeros(128),
                           r.uniform(-0.05, 0.05, 128), np.zeros(1)]).astype(np.float32)


# -------------------------------------------------------------------------- prepare


def _fit_model(case, m12, m13, count):
    import goofit_amd as G
    model = W.build_dalitz(nbins=case["grid"], resonances=_table(case["nres"]))
    data = G.UnbinnedDataSet(model.observables)
    data.from_columns([m12.cpu().numpy(), m13.cpu().numpy(), np.arange(count, dtype=np.float64)])
    return model, data, {k: v.value for k, v in model.params.items()}


def _toy_counts(case, seed):
    r = np.random.default_rng(seed + 21)
    return [int(v) for v in r.integers(case["n"] // 2, case["n"] + 1, case["toys"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("add1d", "prod3d", "mixture"):
        v = _shape_params(case, seed)
        arrays = _flatten(_shape_node(case, v))
        ctx = capi.Context(0)
        ctx.set_program(*arrays)
        ctx.upload_columns([c.cpu().numpy() for c in _shape_columns(case, seed)])
        return dict(case=case, v=v, ctx=ctx, params=arrays[1], norms=arrays[4])
    if kind in ("dalitz_nll", "dalitz_round", "lineshapes"):
        nres = case["nres"]
        m12, m13 = _dalitz_events(case["n"], nres, seed)
        ctx, arrays = _dalitz_context(nres, m12, m13)
        s = dict(case=case, ctx=ctx)
        if kind == "lineshapes":
            c = _moved(nres, seed)
            s.update(params=_with_couplings(arrays[1], c), norms=arrays[4].copy(), c=c,
                     values=torch.empty(case["n"], dtype=F64, device=DEV))
            return s
        ctx.dalitz_cache(0)
        sets = _round_sets(case, seed) if kind == "dalitz_round" else [_moved(nres, seed)]
        norms = []
        for c in sets:
            norms.append(arrays[4].copy())
            norms[-1][1] = _norm(nres, c, 500)
        s.update(params=[_with_couplings(arrays[1], c) for c in sets], norms=norms)
        return s
    if kind == "tddp":
        cols = _td_columns(case, seed)
        arrays = _flatten(_td_node(case, _td_mix(seed)))
        ctx = capi.Context(0)
        ctx.set_program(*arrays)
        ctx.set_decay(DECAY)
        ctx.upload_columns([c.cpu().numpy() for c in cols])
        ctx.set_identity_column(4)
        ctx.dalitz_set_data_size(0, case["n"])
        ctx.dalitz_cache(0)
        norms = arrays[4].copy()
        norms[1] = _td_norm(case)
        return dict(case=case, ctx=ctx, params=arrays[1], norms=norms)
    if kind == "generate":
        c = _moved(case["nres"], seed)
        ctx = capi.Context(0)
        ctx.set_program(*_flatten(_dalitz_node(case["nres"], c)))
        ctx.set_decay(DECAY)
        return dict(case=case, ctx=ctx, seed=seed + 1)
    if kind == "fit":
        m12, m13 = _dalitz_events(case["n"], case["nres"], seed)
        model, data, start = _fit_model(case, m12, m13, case["n"])
        return dict(case=case, model=model, data=data, start=start)
    if kind == "toys":
        counts = _toy_counts(case, seed)
        m12, m13 = _dalitz_events(sum(counts), case["nres"], seed)
        model, data, start = _fit_model(case, m12, m13, sum(counts))
        first = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(int).tolist()
        return dict(case=case, model=model, data=data, start=start, first=first, counts=counts)
    m12, m13 = _dalitz_events(case["n"], 16, seed)
    ctx = capi.Context(0)
    return dict(case=case, ctx=ctx, net=capi.Proposal(ctx, 1, case["batch"]), m12=m12, m13=m13,
                params=_net_params(seed), seed=seed + TRAIN_SEED)


# ------------------------------------------------------------------------------ run


def _shape_norms(s):
    """The normalisations of a likelihood call: analytic where there is an integral, on the grid otherwise."""
    case, v, norms = s["case"], s["v"], s["norms"]
    gauss = v["sigma"] * math.sqrt(2 * math.pi)
    if case["kind"] == "add1d":
        values = {1: gauss, 2: _exp_integral(v["alpha"], -5.0, 5.0)}
    elif case["kind"] == "prod3d":
        values = {1: gauss, 2: _exp_integral(v["alpha"], 0.0, 8.0),
                  3: s["ctx"].reduce_bins(3, [0.0, 10.0, 200.0]) * 10.0 / 200}
    else:
        nb = case["nbins"]
        values = {2: gauss, 3: s["ctx"].reduce_bins(3, [0.0, 10.0, float(nb)]) * 10.0 / nb,
                  5: s["ctx"].reduce_bins(5, [-3.0, 3.0, float(nb)]) * 6.0 / nb,
                  6: _exp_integral(v["slope"], 0.0, 10.0)}
    for f, i in values.items():
        norms[2 * f + 1] = 1.0 / i
    return norms


def run(s):
    case = s["case"]
    kind = case["kind"]
    ctx = s.get("ctx")
    if kind in ("add1d", "prod3d", "mixture"):
        ctx.update_params(s["params"])
        ctx.update_norms(_shape_norms(s))
        return np.array(ctx.reduce_metric("NLL")[0])
    if kind == "dalitz_nll":
        ctx.update_params(s["params"][0])
        ctx.update_norms(s["norms"][0])
        return np.array(ctx.reduce_metric("NLL")[0])
    if kind == "dalitz_round":
        return ctx.reduce_metric_multi("NLL", s["params"], s["norms"])
    if kind == "lineshapes":
        nres, grid = case["nres"], case["grid"]
        ctx.update_params(s["params"])
        ctx.dalitz_cache(0)
        gram = ctx.dalitz_gram(0, [0.0, 3.0, grid, 0.0, 3.0, grid], 1 + nres, nres)
        c = s["c"]
        s["norms"][1] = 1.0 / ((c[:, None] * c.conj()[None, :] * gram).sum().real * (3.0 / grid) ** 2)
        ctx.update_norms(s["norms"])
        ctx.eval_metric_device("NLL", s["values"].data_ptr(), case["n"])
        return dict(gram=gram, values=s["values"])
    if kind == "tddp":
        ctx.update_params(s["params"])
        ctx.update_norms(s["norms"])
        return np.array(ctx.reduce_metric("NLL")[0])
    if kind == "generate":
        m12, m13, tried, top = ctx.dalitz_generate(0, case["n"], s["seed"], BOX)
        return dict(m12=m12, m13=m13, tried=tried, top=np.array(top))
    if kind == "train":
        s["net"].set_params(s["params"])
        first, last = s["net"].train(s["m12"].data_ptr(), s["m13"].data_ptr(), case["n"], BOX, case["steps"],
                                     case["batch"], TRAIN_LR, s["seed"])
        return dict(params=s["net"].get_params(), first=first, last=last)
    import goofit_amd as G
    model = s["model"]
    for k, v in s["start"].items():
        model.params[k].value = v
    model.pdf.setData(s["data"])
    if kind == "fit":
        model.pdf.setDataSize(case["n"])
        fm = G.FitManager(model.pdf)
        fm.setVerbosity(0)
        m = fm.fit()
        free = np.asarray(fm.free_mask(), bool)
        return dict(fval=np.array(m.Fval()), values=np.asarray(m.values())[free], errors=np.asarray(m.errors())[free])
    model.pdf.setDataSize(sum(s["counts"]))
    bf = G.BatchFitter(model.pdf, s["first"], s["counts"])
    bf.fit(threads=case["toys"])
    free = np.asarray(G.FitManager(model.pdf).free_mask(), bool)
    return dict(fval=np.asarray(bf.fval()), values=np.asarray(bf.values())[:, free],
                errors=np.asarray(bf.errors())[:, free])


# ----------------------------------------------------------------------------- work


def work(case):
    """Inputs read once, outputs written once; operations by the formulas (a lineshape about
    150, an exponential or logarithm 20, a complementary error function 40)."""
    kind, n = case["kind"], case.get("n", 0)
    if kind == "add1d":
        return dict(bytes=8.0 * n, flops=75.0 * n)
    if kind == "prod3d":
        return dict(bytes=24.0 * n, flops=130.0 * n)
    if kind == "mixture":
        return dict(bytes=16.0 * n, flops=(150.0 + 2 * case["degree"]) * n + 100.0 * case["nbins"])
    nres = case.get("nres", 16)
    if kind == "dalitz_nll":
        return dict(bytes=16.0 * nres * n, flops=(8.0 * nres + 8) * n)
    if kind == "dalitz_round":
        return dict(bytes=16.0 * nres * n, flops=(8.0 * nres + 8) * n * case["sets"])
    if kind == "lineshapes":
        cells = case["grid"] ** 2 * 0.3  # those inside the plot
        return dict(bytes=(16.0 + 2 * 16 * nres + 8) * n, flops=150.0 * nres * (n + cells) + 8.0 * nres * n
                    + 4.0 * nres * nres * cells)
    if kind == "tddp":
        gauss = 3 * 260.0 if case["threegauss"] else 100.0
        return dict(bytes=(32.0 * nres + (48 if case["mistag"] else 32)) * n,
                    flops=(16.0 * nres + 30 + gauss * (2 if case["mistag"] else 1)) * n)
    if kind == "generate":  # about 20 candidates in the plot for an event
        return dict(bytes=16.0 * n, flops=20 * 158.0 * nres * n)
    if kind == "fit":  # about 30 sweeps over the cache: rounds of 32 sets and single calls
        return dict(bytes=(16.0 + 30 * 16 * nres) * n, flops=600 * 8.0 * nres * n + 150.0 * nres * n)
    if kind == "toys":  # about 15 sweeps over each toy's cache, 300 calls each
        rows = 0.75 * n * case["toys"]
        return dict(bytes=(16.0 + 15 * 16 * nres) * rows, flops=300 * 8.0 * nres * rows)
    return dict(bytes=case["steps"] * (8.0 * case["batch"] + 3 * 4 * 17025 * 2),
                flops=case["steps"] * case["batch"] * 6.0 * 17000)


def tolerance(case):
    """About four times what another order of the sums, or inputs moved by a rounding, was seen to give."""
    kind = case["kind"]
    if kind in ("fit", "toys"):
        # derivative steps turn roundings of the likelihood into differences of MIGRAD's stopping point,
        # which is itself 1e-4 from the minimum
        return dict(rel=1e-5, max=5e-4)
    if kind == "train":
        return dict(rel=1e-3, max=0.1)  # bfloat16 products, Adam's normalised steps
    if kind == "generate":
        return dict(rel=1e-14)  # the same accepted candidates
    if kind == "lineshapes":
        return dict(rel=2e-12, max=1e-10)
    return dict(rel=1e-13)  # 64-bit sums


# ---------------------------------------------------------------------------- exact


def _nll(p):
    return np.array(float(-torch.log(p[p > 0]).sum()))


def _exact_shapes(case, seed):
    v, cols = _shape_params(case, seed), _shape_columns(case, seed)
    gauss = v["sigma"] * math.sqrt(2 * math.pi)
    g = torch.exp(-0.5 * ((cols[0] - v["mu"]) / v["sigma"]) ** 2) / gauss
    if case["kind"] == "add1d":
        e = torch.exp(v["alpha"] * cols[0]) / _exp_integral(v["alpha"], -5.0, 5.0)
        return _nll(v["frac"] * g + (1 - v["frac"]) * e)
    if case["kind"] == "prod3d":
        e = torch.exp(v["alpha"] * cols[1]) / _exp_integral(v["alpha"], 0.0, 8.0)
        i = float(_expgaus(_grid1(0.0, 10.0, 200), 0.0, 0.1, v["rate"]).sum()) * 10.0 / 200
        return _nll(g * e * _expgaus(cols[2], 0.0, 0.1, v["rate"]) / i)

    def poly(x):
        return sum(c * x ** k for k, c in enumerate(v["poly"]))
    nb = case["nbins"]
    it = float(_expgaus(_grid1(0.0, 10.0, nb), 0.0, 0.1, v["rate"]).sum()) * 10.0 / nb
    ip = float(poly(_grid1(-3.0, 3.0, nb)).sum()) * 6.0 / nb
    sig = g * _expgaus(cols[1], 0.0, 0.1, v["rate"]) / it
    bkg = poly(cols[0]) / ip * torch.exp(v["slope"] * cols[1]) / _exp_integral(v["slope"], 0.0, 10.0)
    return _nll(v["frac"] * sig + (1 - v["frac"]) * bkg)


def _td_terms(R, tau, t, x, y, sigma):
    """The cosh, cos, sinh, sin terms of the three-Gaussian resolution."""
    fc, ft = R[0], R[1]
    parts = ((fc, R[2] + R[9], R[3] * R[10]), (ft, R[4] + R[11], R[5] * R[12]),
             (1 - fc - ft, R[6] + R[11], R[7] * R[12]))
    out = [0, 0, 0, 0]
    for f, bias, scale in parts:
        tt, s = t - bias * sigma, scale * sigma
        a1, g = s * math.sqrt(2.0), 1 / tau
        a2, b, c = 0.5 * a1, g - tt / (s * s), 0.5 * tt * tt / (s * s)
        ng, rp = math.sqrt(0.5 / math.pi) / s, math.sqrt(math.pi) / 2
        u = a2 * (b + R[8])
        big = a1 * torch.exp(u * u - c)
        i0 = rp * torch.erfc(u)
        i1 = 0.5 * torch.exp(-u * u)
        i2 = i1 * u + 0.5 * i0
        i3 = i1 * (u * u + 1)
        r = x * g * a1
        j0 = big * i0
        j1 = big * r * (i1 - u * i0)
        j2 = big * r * r * (i2 - 2 * u * i1 + u * u * i0)
        j3 = big * r ** 3 * (i3 - 3 * u * i2 + 3 * u * u * i1 - u ** 3 * i0)
        up, um = a2 * (b - y * g + R[8]), a2 * (b + y * g + R[8])
        ip = a1 * torch.exp(up * up - c) * rp * torch.erfc(up)
        im = a1 * torch.exp(um * um - c) * rp * torch.erfc(um)
        for k, v in enumerate((ng * 0.5 * (ip + im), ng * (j0 - 0.5 * j2), ng * 0.5 * (ip - im), ng * (j1 - j3 / 6))):
            out[k] = out[k] + f * v
    return out


def _exact_tddp(case, seed):
    cols, mix = _td_columns(case, seed), _td_mix(seed)
    t, s, m12, m13 = cols[:4]
    c = _couplings(case["nres"])
    a, b = _amplitude(case["nres"], c, m12, m13), _amplitude(case["nres"], c, m12, m13, swap=True)
    na, nb, ab = a.abs().square(), b.abs().square(), a * b.conj()
    t1, t2 = na + nb, na - nb

    def rate(tau, x, y, sign):
        if case["threegauss"]:
            p = _td_terms(TG, tau, t, x, y, s)
            return t1 * p[0] + sign * t2 * p[1] - 2 * ab.real * p[2] - 2 * sign * ab.imag * p[3]
        d = t / tau
        return (t1 * torch.cosh(y * d) + sign * t2 * torch.cos(x * d) - 2 * ab.real * torch.sinh(y * d)
                - 2 * sign * ab.imag * torch.sin(x * d)) * torch.exp(-d)
    v = rate(mix[0], mix[1], mix[2], 1)
    if case["mistag"]:
        w = cols[5]
        v = torch.where(w > 0, (1 - 2 * w) * v + w * rate(0.4101, 0.0039, 0.0065, -1) + w * rate(0.4101, 0.0039, 0.0065, 1), v)
    return _nll(v * _td_norm(case))


def _mix64(z):
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _unif(key, counter):
    return (_mix64(np.uint64(key) ^ _mix64(counter)) >> np.uint64(11)).astype(np.float64) / 9007199254740992.0


def _exact_generate(case, seed):
    """The documented stream: uniform candidates by counter, kept where u fmax < |A|^2."""
    c, n = _moved(case["nres"], seed), case["n"]
    pass_ = 1 << 22
    with np.errstate(over="ignore"):
        key = _mix64(np.array([seed + 1], np.uint64) ^ np.uint64(0x6A09E667F3BCC909))[0]

        def candidates(base):
            k = np.arange(base, base + pass_, dtype=np.uint64)
            p = [torch.as_tensor(0.0 + _unif(key, np.uint64(2) * k + np.uint64(j)) * 3.0, device=DEV) for j in (0, 1)]
            v = torch.zeros(pass_, dtype=F64, device=DEV)
            ok = _inside(*p)
            v[ok] = _amplitude(case["nres"], c, p[0][ok], p[1][ok]).abs().square()
            return p[0], p[1], v, torch.as_tensor(_unif(key ^ np.uint64(0xD1B54A32D192ED03), k), device=DEV)
        top = 1.25 * float(candidates(0)[2].max())
        base, got = pass_, []
        while sum(g.shape[1] for g in got) < n:
            m12, m13, v, u = candidates(base)
            take = u * top < v
            got.append(torch.stack([m12[take], m13[take]]))
            base += pass_
    m = torch.cat(got, 1)[:, :n].cpu().numpy()
    return dict(m12=m[0], m13=m[1], tried=base, top=np.array(top))


def _newton(w, integrals, area, c, free):
    """The minimum of -sum log(|c w|^2 / norm) over the couplings `free`: its value and place."""
    n = w.shape[1]
    z = torch.as_tensor(c, device=DEV)
    real = torch.cat([w, 1j * w])  # d(amplitude) / d(re c), d / d(im c)
    basis = torch.cat([torch.eye(len(c), dtype=torch.complex128, device=DEV), 1j * torch.eye(len(c), dtype=torch.complex128, device=DEV)])
    m = basis @ integrals @ basis.conj().T.contiguous() * area
    m = m.real.contiguous()
    x = torch.cat([z.real, z.imag])
    for _ in range(12):
        a = (torch.complex(x[:len(c)], x[len(c):])[:, None] * w).sum(0)
        p = a.abs().square()
        g = 2 * (real * a.conj()).real / p
        norm = x @ m @ x
        d = m @ x
        grad = -g.sum(1) + n * 2 * d / norm
        r2 = real / a.abs()
        hess = g @ g.T.contiguous() - 2 * (r2 @ r2.conj().T.contiguous()).real + n * (2 * m / norm - 4 * torch.outer(d, d) / norm ** 2)
        f = torch.as_tensor(free, device=DEV)
        cov = torch.linalg.inv(hess[f][:, f])
        step = cov @ grad[f]
        x = x.clone()
        x[f] -= step
    keep = [k for i in range(len(c)) for k in (i, len(c) + i) if k in free]  # re, im of each in turn
    a = (torch.complex(x[:len(c)], x[len(c):])[:, None] * w).sum(0)
    fval = float(-torch.log(a.abs().square() / (x @ m @ x)).sum())
    return fval, x[keep].cpu().numpy()


def _exact_fits(case, seed):
    nres = case["nres"]
    counts = _toy_counts(case, seed) if case["kind"] == "toys" else [case["n"]]
    m12, m13 = _dalitz_events(sum(counts), nres, seed)
    integrals = _integrals(nres, case["grid"])
    free = [k for k in range(2 * nres) if k % nres != 1]  # the second resonance's coupling is held
    out, at = [], 0
    for k in counts:
        w = _waves(nres, m12[at:at + k], m13[at:at + k])
        out.append(_newton(w, integrals, (3.0 / case["grid"]) ** 2, _couplings(nres), free))
        at += k
    # MIGRAD's errors are numerical estimates, so only the minimum has a value of its own
    if case["kind"] == "fit":
        return dict(fval=np.array(out[0][0]), values=out[0][1], errors=None)
    return dict(fval=np.array([o[0] for o in out]), values=np.stack([o[1] for o in out]), errors=None)


def _exact_train(case, seed):
    """The training in 64 bits: the documented batches, loss and Adam steps."""
    m12, m13 = _dalitz_events(case["n"], 16, seed)
    data = torch.stack([m12, m13]) / 3.0
    h, half, key0 = 128, case["batch"] // 2, seed + TRAIN_SEED
    p = torch.as_tensor(_net_params(seed).astype(np.float64), device=DEV).requires_grad_(True)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    losses = []
    with np.errstate(over="ignore"):
        for k in range(case["steps"]):
            key = np.uint64((key0 * 0x9E3779B97F4A7C15 + 2 * k + 1) % 2 ** 64)
            i = np.arange(case["batch"], dtype=np.uint64)
            e = _mix64(key ^ _mix64(np.uint64(2) * i[:half])) % np.uint64(case["n"])
            uv = np.stack([_unif(key + np.uint64(1), np.uint64(2) * i[half:] + np.uint64(j)) for j in (0, 1)])
            xy = torch.cat([data[:, torch.as_tensor(e.astype(np.int64), device=DEV)],
                            torch.as_tensor(uv, device=DEV)], 1) * 2 - 1
            w1, b1 = p[:2 * h].view(h, 2), p[2 * h:3 * h]
            w2 = p[3 * h:3 * h + h * h].view(h, h)
            b2, w3, b3 = p[-2 * h - 1:-h - 1], p[-h - 1:-1], p[-1]
            z1 = w1 @ xy + b1[:, None]
            z2 = w2 @ (z1 * torch.sigmoid(z1)) + b2[:, None]
            f = w3 @ (z2 * torch.sigmoid(z2)) + b3
            loss = -f[:half].mean() + torch.logsumexp(f[half:], 0) - math.log(half)
            losses.append(float(loss))
            g, = torch.autograd.grad(loss, p)
            lr = TRAIN_LR * (0.05 + 0.95 * 0.5 * (1 + math.cos(math.pi * k / case["steps"])))
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            step = lr * (m / (1 - 0.9 ** (k + 1))) / (torch.sqrt(v / (1 - 0.999 ** (k + 1))) + 1e-8)
            p = (p.detach() - step).requires_grad_(True)
    return dict(params=p.detach().cpu().numpy(), first=losses[0], last=losses[-1])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("add1d", "prod3d", "mixture"):
        return _exact_shapes(case, seed)
    if kind == "tddp":
        return _exact_tddp(case, seed)
    if kind == "generate":
        return _exact_generate(case, seed)
    if kind in ("fit", "toys"):
        return _exact_fits(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    nres = case["nres"]
    m12, m13 = _dalitz_events(case["n"], nres, seed)
    if kind == "dalitz_nll":
        c = _moved(nres, seed)
        return _nll(_amplitude(nres, c, m12, m13).abs().square() * _norm(nres, c, 500))
    if kind == "dalitz_round":
        sets = _round_sets(case, seed)
        w = torch.cat([_waves(nres, x, y) for x, y in zip(m12.split(CHUNK), m13.split(CHUNK))], 1)
        base = (torch.as_tensor(sets[0], device=DEV)[:, None] * w).sum(0)
        out = []
        for c in sets:
            d = c - sets[0]
            a = base + sum(complex(d[j]) * w[j] for j in np.nonzero(d)[0])
            out.append(_nll(a.abs().square() * _norm(nres, c, 500)))
        return np.array(out)
    c = _moved(nres, seed)
    gram = _integrals(nres, case["grid"]).cpu().numpy()
    norm = 1.0 / ((c[:, None] * c.conj()[None, :] * gram).sum().real * (3.0 / case["grid"]) ** 2)
    return dict(gram=gram, values=-torch.log(_amplitude(nres, c, m12, m13).abs().square() * norm))
