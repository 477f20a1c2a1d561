"""GPU test of coefficient solves that level space cannot finish: a y that the
FEs explain in full (what a regression passes), with and without FEs that are
collinear, at the default tolerance and a tight one, and a NaN in y.  Through
every coefficient entry point, on a fresh handle and on one that solved another
column before, against the passes over the observations (FEHIP_NORMAL=0).

Coefficients are compared by their fit: at tol 1e-12 both sides' fits are
determined to about 1e-10 (tests/test_gpu_level_space.py), at 1e-8 to 1e-8
times the condition (below 30 here); the bars are ten times and more above."""
import numpy as np
import pytest

from fixedeffects_rocm import api, warmstart

pytestmark = pytest.mark.gpu

BAR = {1e-12: 1e-9, 1e-8: 1e-5}


def _refs(shape, rng):
    if shape == "two_way":
        return [rng.integers(1, 301, 5_003), rng.integers(1, 41, 5_003)]
    if shape == "network":
        a = rng.integers(0, 800, 8_009)
        return [a + 1, np.clip(a // 8 + rng.integers(-6, 7, 8_009), 0, 99) + 1]
    if shape == "twice":
        r = rng.integers(1, 301, 5_003)
        return [r, rng.integers(1, 41, 5_003), r.copy()]
    if shape == "constant":
        return [rng.integers(1, 1_001, 20_011), np.ones(20_011, np.int64)]
    if shape == "grid":
        a, b, c = np.meshgrid(np.arange(20), np.arange(30), np.arange(7), indexing="ij")
        return [a.ravel() + 1, b.ravel() + 1, c.ravel() + 1]
    return [rng.integers(1, 9, 400), rng.integers(1, 6, 400)]  # "few"


def _problem(shape):
    rng = np.random.default_rng(11)
    refs = [np.asarray(r, np.int64) for r in _refs(shape, rng)]
    n = [int(r.max()) for r in refs]
    fit = sum(rng.standard_normal(k)[r - 1] for r, k in zip(refs, n))
    return refs, n, fit, rng


def _fit(blocks, refs):
    return sum(b[r - 1] for b, r in zip(blocks, refs))


def _solve(entry, s, refs, n, y, tol, maxiter=1_000):
    """The fit of the returned coefficients, and whether the solve converged."""
    if entry == "full":
        obs, _, cv = s.solve_coefficients(y, tol=tol, maxiter=maxiter)
        return sum(obs), cv
    if entry == "levels":
        _, blocks, _, cv = s.solve_coefficients_full(y, tol=tol, maxiter=maxiter, per_obs=False)
    elif entry == "raw":
        blocks, _, cv = s.solve_coefficients_raw(y, tol=tol, maxiter=maxiter)
    else:
        start = np.random.default_rng(3).standard_normal(sum(n))
        blocks, _, cv = warmstart.solve_coefficients_from(s, y, start, tol=tol, maxiter=maxiter)
    return _fit(blocks, refs), cv


def _handle(monkeypatch, on, refs, n, precision, algorithm, w=None):
    monkeypatch.setenv("FEHIP_NORMAL", on)
    return api.FixedEffectSolverROCm([api.FixedEffect.from_refs(r, k) for r, k in zip(refs, n)], w, precision,
                                     algorithm=algorithm)


@pytest.mark.parametrize("shape", ["two_way", "network", "twice", "constant", "grid", "few"])
@pytest.mark.parametrize("algorithm", ["lsmr", "projected"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("entry", ["full", "levels", "raw", "x0"])
def test_explained(gpu, monkeypatch, entry, precision, algorithm, shape):
    refs, n, fit, rng = _problem(shape)
    w = rng.lognormal(0, 0.5, len(fit)) if shape in ("network", "grid") else None
    other = 5.0 * rng.standard_normal(len(fit))
    for tol, bar in BAR.items():
        for y in (fit, fit + rng.standard_normal(len(fit))):
            with _handle(monkeypatch, "0", refs, n, "fp64", algorithm, w) as s:
                want, ok = _solve(entry, s, refs, n, y, tol)
            with _handle(monkeypatch, "1", refs, n, precision, algorithm, w) as s:
                got = [_solve(entry, s, refs, n, y, tol)]
                s.solve_residuals(other.copy(), tol=tol, maxiter=1_000)
                got.append(_solve(entry, s, refs, n, y, tol))
            for f, cv in got:
                assert np.linalg.norm(f - want) <= bar * np.linalg.norm(y)
                assert precision == "mixed" or cv == ok  # (the mixed mode aims at a tolerance of its own)


@pytest.mark.parametrize("algorithm", ["lsmr", "projected"])
@pytest.mark.parametrize("entry", ["full", "raw", "x0"])
def test_nan(gpu, monkeypatch, entry, algorithm):
    refs, n, fit, rng = _problem("two_way")
    fit[17] = np.nan
    out = []
    for on in ("1", "0"):
        with _handle(monkeypatch, on, refs, n, "fp64", algorithm) as s:
            s.solve_residuals(rng.standard_normal(len(fit)), maxiter=100)
            out.append(_solve(entry, s, refs, n, fit, 1e-8, maxiter=100))
    assert np.array_equal(out[0][0], out[1][0], equal_nan=True) and out[0][1] == out[1][1]
