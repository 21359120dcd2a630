"""The kernel of a lone time-dependent Dalitz node (k_td_reduce) against the interpreter, and
the three-Gaussian decay-time terms against 60-digit arithmetic."""
import math

import mpmath
import numpy as np
import pytest

import oracle as O
from goofit_amd import capi
from goofit_amd import workloads as W

from _models import arrays, tddp, tddp_events, threegauss

pytestmark = pytest.mark.gpu

MIX = (0.4101, 0.012, 0.02, 0.004, -0.003)


def _load(ctx, top, aos):
    ctx.set_program(*arrays(top)[1])
    ctx.set_decay(W.DALITZ_DECAY)
    ctx.upload_columns([np.ascontiguousarray(aos[:, k]) for k in range(aos.shape[1])])
    ctx.set_identity_column(4)
    ctx.dalitz_set_data_size(top.function_idx, len(aos))
    ctx.dalitz_cache(top.function_idx)


@pytest.mark.parametrize("kind", ["truth", "threegauss"])
@pytest.mark.parametrize("n,nres,tags", [(1, 1, False), (255, 4, True), (257, 5, False), (3000, 8, True),
                                         (3001, 9, False), (200_003, 16, True)])
def test_lone_node_kernel_equals_interpreter(ctx, kind, n, nres, tags):
    """Events at the edges of a workgroup, resonances at the edges of its chunks of four, with
    and without mistag and tag columns.  Each event's value has the same
    bits on both paths and the factors only meet in another order: n roundings of 2^-53 in
    the product, taken by chance, stay below 4 sqrt(n) 2^-53 of a sum of n logarithms."""
    rng = np.random.default_rng(n + nres)
    kw = dict(mistag=rng.uniform(-0.1, 0.3, n), tag=rng.choice([-1.0, 1.0, 0.0], n)) if tags else {}
    top, _ = tddp(mix=MIX, resonances=W.DALITZ_RESONANCES[:nres], mistag=tags, charmtag=tags,
                    resolution=threegauss() if kind == "threegauss" else O.TruthResolution())
    aos = tddp_events(n, seed=n, **kw)
    if n == 1:
        aos[0, 2:4] = 1.0, 1.0  # inside
    _load(ctx, top, aos)
    for metric in ("NLL", "PROB"):
        got = {}
        for knob in (1, 0):
            ctx.set_tuning(capi.TUNE_FAST_DALITZ, knob)
            got[knob] = ctx.reduce_metric(metric)[0]
        ctx.set_tuning(capi.TUNE_FAST_DALITZ, 1)
        assert got[0] != 0 and math.isfinite(got[0])
        assert abs(got[1] - got[0]) <= 4 * (1 + math.sqrt(n)) * 2.0**-53 * max(abs(got[0]), n), (metric, got)


def test_time_terms_exact(ctx):
    """Each event's rate at decay times from 5 widths before 0 to 400 widths after it, from the
    cached waves in 60 digits.  With q = width / lifetime and w = time / width the tails'
    exponent q w and, before the peak, w^2 carry a few roundings each: 4 units of 2^-53 of
    either, and 40 for the sums.  (exp(u^2 - w^2 / 2), formed from the difference, is off by w^2 / 2
    of them: 80000 at 400 widths.)"""
    times = np.array([-0.25, -0.1, -0.03, 0.0, 0.004, 0.05, 0.2, 0.7, 2.0, 6.0, 20.0])
    top, _ = tddp(mix=MIX, resonances=W.DALITZ_RESONANCES[:1], resolution=threegauss())
    aos = np.array([[t, 0.05, 1.0, 0.9, i] for i, t in enumerate(times)])
    _load(ctx, top, aos)
    coup = [complex(r.amp_real.value, r.amp_imag.value) for r in top.resonances]
    R = [float(v.value) for v in top.resolution.params]
    a = ctx.dalitz_get_cache(top.function_idx, 0, len(times))
    b = ctx.dalitz_get_cache(top.function_idx, 1, len(times))
    got = ctx.eval_metric("EVAL")
    with mpmath.workdps(60):
        f = [mpmath.mpf(v) for v in R]
        tau, x, y = (mpmath.mpf(v) for v in MIX[:3])
        shapes = [(f[0], f[2] + f[9], f[3] * f[10]), (f[1], f[4] + f[11], f[5] * f[12]),
                  (1 - f[0] - f[1], f[6] + f[11], f[7] * f[12])]
        for i, t in enumerate(times):
            A, B = (mpmath.mpc(coup[0]) * mpmath.mpc(complex(v[i])) for v in (a, b))
            sg, P, units = mpmath.mpf(0.05), [mpmath.mpf(0)] * 4, 40.0
            for frac, bias, scale in shapes:
                s, tt = scale * sg, mpmath.mpf(float(t)) - bias * sg
                w, g0 = tt / s, 1 / tau + f[8]

                def tail(g):
                    q = s * g
                    u = (q - w) / mpmath.sqrt(2)
                    return mpmath.exp(q * (q / 2 - w)) * mpmath.erfc(u)
                S, Sp, Sm = tail(g0), tail(g0 - y / tau), tail(g0 + y / tau)
                u = (s * g0 - w) / mpmath.sqrt(2)
                h = mpmath.exp(-w * w / 2) / (2 * mpmath.sqrt(mpmath.pi))
                r = mpmath.sqrt(2) * s * x / tau
                j2 = S / 2 * (mpmath.mpf(1) / 2 + u * u) - u * h
                j3 = h * (1 + u * u) - u * S / 2 * (mpmath.mpf(3) / 2 + u * u)
                for k, v in enumerate(((Sp + Sm) / 4, S / 2 - r * r / 2 * j2, (Sp - Sm) / 4,
                                       r * (h - u * S / 2 - r * r / 6 * j3))):
                    P[k] += frac * v
                units = max(units, 40 + 4 * abs(float(s * g0 * w)) + (4 * float(w * w) if w < 0 else 0))
            nA, nB, AB = abs(A) ** 2, abs(B) ** 2, A * mpmath.conj(B)
            ref = (nA + nB) * P[0] + (nA - nB) * P[1] - 2 * AB.real * P[2] - 2 * AB.imag * P[3]
            assert abs(float(got[i] / ref - 1)) < units * 2.0**-53, (t, got[i], float(ref))
