"""Pins the symmetric segment math of the fused kernels and the register row
kernel on the CPU.

seg_mean_tilt, seg_shares_h and seg_shares_grad_h (csrc/ca_common.h) are
re-evaluated here in float32 numpy, with the polynomial (CA_TILT), the switch
point (kHalfSeriesT) and the factor 4 (kShareShift) parsed from the header, and
compared with the float64 oracle's segment terms, as tests/test_device_math.py
does for the one-sided forms.  A wrong coefficient, switch point, sign or factor
fails these checks without a GPU.
"""
import math
import re

import numpy as np
import pytest

from test_device_math import HDR, coeffs, f32, poly, reference_terms

HALF_LN2 = f32(0.34657359027997265)
EPS = 2.0 ** -24


def constant(name):
    return f32(float(re.search(r"%s = ([0-9.e-]+)f" % name, open(HDR).read()).group(1)))


H_SW = float(constant("kHalfSeriesT"))


def symmetric_terms(sl, sr, pl, pr, gl=None, gr=None, tilt=None, switch=None, sign=1):
    """float32 restatement of seg_shares_h / seg_shares_grad_h: (4L, 4R) and,
    with gradients, (4 dL, 4 dR)."""
    sl, sr, pl, pr = (np.asarray(v, f32) for v in (sl, sr, pl, pr))
    h = (sr - sl) * HALF_LN2
    dp, sp = pr - pl, pr + pl
    with np.errstate(divide="ignore", invalid="ignore"):
        inv_h = f32(1) / h
        ac = dp * inv_h
        dc = (sp - ac) * inv_h
        bc = dc * inv_h
    c = poly(h * h, coeffs("CA_TILT") if tilt is None else tilt)
    ds = f32(sign) * dp * c
    as_ = sp - h * ds
    bs = as_ * c
    small = np.abs(h) < f32(H_SW if switch is None else switch)
    a, d = np.where(small, as_, ac), np.where(small, ds, dc)
    L, R = a - d, a + d
    if gl is None:
        return L, R
    t = (gr - gl) * np.where(small, bs, bc)
    return L, R, gl * L + t, gr * R - t


@pytest.fixture(scope="module")
def grid():
    rng = np.random.default_rng(11)
    edge = 2 * H_SW / math.log(2)  # the switch in log2 score differences
    d = np.concatenate([np.linspace(-60, 60, 6001), np.linspace(-3, 3, 2001),
                        [0.0, 1e-7, -1e-7, 1e-4, -1e-4],
                        edge + np.linspace(-1e-3, 1e-3, 41), -edge + np.linspace(-1e-3, 1e-3, 41)])
    base = rng.uniform(-9, 7, d.size)
    sl, sr = base.astype(f32), (base + d).astype(f32)
    keep = (sl <= 8) & (sr <= 8)  # kernels keep s - m <= 8
    return sl[keep], sr[keep]


def reference(sl, sr, gl, gr):
    L, R, J2, E = reference_terms(sl.astype(np.float64), sr.astype(np.float64), 0.0)
    x = R - J2  # weight of u (1 - u)
    return L, R, gl * (L - x) + gr * x, gl * x + gr * J2, E


def errors(sl, sr, **kw):
    rng = np.random.default_rng(12)
    gl, gr = (rng.standard_normal(sl.size).astype(f32) for _ in range(2))
    got = symmetric_terms(sl, sr, np.exp2(sl), np.exp2(sr), gl, gr, **kw)
    *ref, E = reference(sl, sr, gl.astype(np.float64), gr.astype(np.float64))
    scale = (E, E, E * (np.abs(gl) + np.abs(gr)), E * (np.abs(gl) + np.abs(gr)))
    return [np.max(np.abs(a.astype(np.float64) / 4 - b) / s) for a, b, s in zip(got, ref, scale)]


def test_shares_and_gradients_match_oracle(grid):
    """Errors relative to the segment's larger endpoint weight E.  The endpoint
    weights and h carry an ulp each; just above the switch dp / h, of size 2 E,
    loses 1 / h of its relative error twice over: about (1 + 1 / h^2) ulp of E,
    in shares a quarter of that."""
    bound = (1 + 1 / H_SW ** 2) * 4 * EPS
    err = errors(*grid)
    assert max(err[:2]) < bound and max(err[2:]) < bound, (err, bound)
    L, R = symmetric_terms(*grid, np.exp2(grid[0]), np.exp2(grid[1]))
    assert np.all(np.isfinite(L)) and np.all(np.isfinite(R)) and np.all(L >= 0) and np.all(R >= 0)


def test_continuous_at_the_switch_and_exact_at_equal_scores():
    s = np.linspace(-5, 5, 101).astype(f32)
    p = np.exp2(s)
    L, R = symmetric_terms(s, s, p, p)
    assert np.array_equal(L, 2 * p) and np.array_equal(R, 2 * p)  # 4 L = 4 (p / 2)
    d = f32(2 * H_SW / math.log(2))
    for sign in (1, -1):
        out = [symmetric_terms(s, s + f32(sign) * d, p, np.exp2(s + f32(sign) * d), switch=t)
               for t in (0.0, 1.0)]  # quotients, series
        for a, b in zip(*out):
            assert np.max(np.abs(a - b) / np.maximum(p, np.exp2(s + f32(sign) * d))) < 64 * EPS


def test_tilt_polynomial():
    """CA_TILT against C(y) = (coth h - 1/h) / h, y = h^2, from its power series
    (1/3 - y/45 + 2y^2/945 - y^3/4725 + 2y^4/93555 - ...): the stated 1.5e-7
    relative error."""
    c = [float(v) for v in coeffs("CA_TILT")]
    for h in np.linspace(1e-3, H_SW, 200):
        y = h * h
        ref = 1 / 3 - y / 45 + 2 * y ** 2 / 945 - y ** 3 / 4725 + 2 * y ** 4 / 93555 - 1382 * y ** 5 / 638512875
        assert abs(c[0] + c[1] * y + c[2] * y * y - ref) / ref < 1.5e-7, h


def test_share_factor_is_four():
    """kShareShift: the kernels take p a factor 2^kShareShift smaller."""
    assert 2.0 ** float(constant("kShareShift")) == 4.0


def test_planted_mistakes_are_caught(grid):
    good = coeffs("CA_TILT")
    clean = max(errors(*grid))
    for kw in (dict(sign=-1), dict(tilt=[good[0], -good[1], good[2]]),
               dict(tilt=[good[0], good[1], f32(0)]), dict(switch=2.0), dict(switch=0.01)):
        assert max(errors(*grid, **kw)) > 3 * clean, kw
