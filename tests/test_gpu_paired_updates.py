"""GPU test of where the level-space iteration may stop when it updates x for
two iterations at once (csrc/normal.hip): after either one of a pair, at any
iteration limit, by a rule with and without ||x||, columns apart from another.
Against the passes over the observations (FEHIP_NORMAL=0), which update x in
each.  Both are at the same iterate, so they differ by rounding alone, which a
few dozen iterations leave far below 1e-9 of the column."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu


def _solve(monkeypatch, on, fes, w, Y, **kw):
    monkeypatch.setenv("FEHIP_NORMAL", on)
    cols = [y.copy() for y in Y]
    with api.FixedEffectSolverROCm(fes, w, "fp64") as s:
        _, it, cv = s.solve_residuals_many(cols, **kw)
        info = [s.lsmr_info(c) for c in range(len(Y))]
    return cols, it, cv, info


@pytest.mark.parametrize("K", [16, 32])  # more than 2048 partials a launch
@pytest.mark.parametrize("tol,maxiter", [(1e-12, m) for m in range(1, 9)] + [(t, 1000) for t in (1e-2, 1e-4, 1e-6)])
def test_stops(gpu, monkeypatch, K, tol, maxiter):
    rng = np.random.default_rng(K)
    N = 30_011
    n = (3_000, 400, 9)
    refs = [rng.integers(0, k, N) for k in n]
    fes = [api.FixedEffect.from_refs(r + 1, k) for r, k in zip(refs, n)]
    w = rng.lognormal(0, 0.5, N)
    Y = []
    for c in range(K):
        fit = sum(rng.standard_normal(k)[r] for r, k in zip(refs, n))
        # noise alone, less and less of it, none (the rules on ||r||), one level's dummy, nothing
        y = [rng.standard_normal(N), fit + 10.0 ** -c * rng.standard_normal(N), fit, 1.0 * (refs[1] == c),
             np.zeros(N)][c % 5]
        Y.append(y)
    a, ia, ca, fa = _solve(monkeypatch, "1", fes, w, Y, tol=tol, maxiter=maxiter)
    b, ib, cb, fb = _solve(monkeypatch, "0", fes, w, Y, tol=tol, maxiter=maxiter)
    assert ia == ib and ca == cb
    for c in range(K):
        assert fa[c]["istop"] == fb[c]["istop"]
        assert np.linalg.norm(a[c] - b[c]) <= 1e-9 * max(np.linalg.norm(Y[c]), 1e-300)
        assert abs(fa[c]["normx"] - fb[c]["normx"]) <= 1e-9 * abs(fb[c]["normx"])
