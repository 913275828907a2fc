"""gelu_erf (csrc/qa_internal.h): the fitted tail polynomial against the exact
GELU in 64 bits, evaluated in f32 as the kernel does, next to the form it
replaces, erf from Abramowitz & Stegun 7.1.26 (src/shaders.rs:2593-2625).  In no
band of x may the largest error be above that form's, absolute or relative.
The coefficients are read from the source."""
from __future__ import annotations

import os
import re

import numpy as np
import pytest
from scipy.special import erfc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F = np.float32


def _fma(a, b, c):
    return (a.astype(np.float64) * np.float64(b) + np.float64(c)).astype(F) if np.isscalar(b) else \
        (a.astype(np.float64) * b.astype(np.float64) + np.float64(c)).astype(F)


def _coefficients():
    text = open(os.path.join(ROOT, "qwen3-aligner-wgpu_amd", "csrc", "qa_internal.h")).read()
    body = text[text.index("float gelu_erf(float x)"):]
    body = body[: body.index("asm(")]
    return [F(c) for c in re.findall(r" (-?\d[\d.]*(?:e-?\d+)?)f\b", body)]


def _tail(x, q):
    """max(x, 0) - |x| q with one rounding."""
    return (np.maximum(x, 0).astype(np.float64) - np.abs(x).astype(np.float64) * q.astype(np.float64)).astype(F)


def _fitted(x):
    ax, cs = np.abs(x), _coefficients()
    p = np.full_like(x, cs[0])
    for c in cs[1:]:
        p = _fma(p, ax, c)
    return _tail(x, np.exp2(p.astype(np.float64)).astype(F))


def _as7126(x):
    t = (F(1) / _fma(np.abs(x), F(0.3275911 * 0.5 ** 0.5), 1.0)).astype(F)
    e = np.exp2((x * x * F(-0.5 * np.log2(np.e))).astype(np.float64)).astype(F)
    p = np.full_like(x, F(0.5 * 1.061405429))
    for c in (-1.453152027, 1.421413741, -0.284496736, 0.254829592):
        p = _fma(p, t, F(0.5 * c))
    return _tail(x, p * t * e)


def _errors(fn, x):
    exact = 0.5 * x.astype(np.float64) * erfc(-x.astype(np.float64) / np.sqrt(2.0))
    err = np.abs(fn(x).astype(np.float64) - exact)
    return err.max(), (err / np.abs(exact)).max()


BANDS = [1e-4, 1e-3, 0.01, 0.03, 0.1, 0.2, 0.5, 1, 2, 3, 4, 5, 5.5, 7, 10]


def test_constant_term_is_exact():
    assert len(_coefficients()) == 11 and _coefficients()[-1] == -1.0


@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("lo,hi", list(zip(BANDS, BANDS[1:])))
def test_no_band_is_further_off_than_7_1_26(lo, hi, sign):
    x = (sign * np.linspace(lo, hi, 40001)).astype(F)
    got, bar = _errors(_fitted, x), _errors(_as7126, x)
    # (above 3 both are the result's rounding, half an ulp of x)
    half_ulp = np.spacing(F(hi)) / 2 if sign > 0 else 0.0
    assert got[0] <= max(bar[0], half_ulp * 1.05) and got[1] <= max(bar[1], half_ulp * 1.05 / lo), (got, bar)


def test_coefficients_solve_the_fit():
    """How they were found: the linear program for the degree-10 polynomial, its
    constant term -1, with the smallest largest ratio of the error in |x| q to
    7.1.26's largest in the same band (the smaller of its absolute and its
    relative one, 0.7 of that past 4, at least 3e-9 x below 1, where f32 rounds
    more).  Its optimum is 0.24; rounded to f32 the coefficients keep 0.34."""
    from scipy.optimize import linprog
    from scipy.special import log_ndtr, ndtr
    a = np.concatenate([np.geomspace(1e-3, 0.2, 300), np.linspace(0.2, 10, 1500)])
    q = ndtr(-a)
    t = 1 / (1 + 0.3275911 * a / np.sqrt(2))
    old = 0.5 * t * np.exp(-a * a / 2) * np.polyval([1.061405429, -1.453152027, 1.421413741, -0.284496736, 0.254829592], t)
    bar = np.empty_like(a)
    for lo, hi in zip(BANDS[1:], BANDS[2:-1] + [11]):
        m = (a >= lo) & (a < hi)
        bar[m] = np.minimum((a * np.abs(old - q))[m].max(), (a * q)[m] * np.abs(old / q - 1)[m].max())
    bar = np.maximum(bar, np.where(a < 1, 3e-9 * a, 0)) * np.where(a > 4, 0.7, 1)
    w = a * q * np.log(2) / bar
    scale = 10.0 ** np.arange(1, 11)  # of the unknowns, for the solver
    rows = w[:, None] * np.stack([a ** k for k in range(1, 11)], 1) / scale
    rhs = w * (log_ndtr(-a) / np.log(2) + 1)
    one = np.ones((len(a), 1))
    best = linprog(np.r_[np.zeros(10), 1], A_ub=np.block([[rows, -one], [-rows, -one]]), b_ub=np.r_[rhs, -rhs],
                   bounds=[(None, None)] * 10 + [(0, None)], method="highs").x[-1]
    mine = np.array(_coefficients(), np.float64)[::-1][1:]
    assert np.abs(rows @ (mine * scale) - rhs).max() <= 0.35 and best < 0.25


def test_falls_past_the_fit():
    """Past 10 the polynomial keeps falling (its leading coefficient is
    negative), to an exponent that gives a zero: no value comes back up."""
    a = np.geomspace(10, 1e38, 4000).astype(F)
    with np.errstate(over="ignore"):
        p = np.full_like(a, _coefficients()[0])
        for c in _coefficients()[1:]:
            p = _fma(p, a, c)
        assert (p <= -76).all() and (np.diff(p[np.isfinite(p)]) <= 0).all()
        assert (_fitted(-a[(a > 40) & (a < 1e30)]) == 0).all()
