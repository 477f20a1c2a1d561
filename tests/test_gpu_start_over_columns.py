"""GPU test of batches in which level space loses some columns (the FEs explain
them in full): those start over on the observations in a batch of their own,
up to half of the columns; the others' results are bit for bit those of a batch
without them.  The columns that start over against the passes over the
observations (FEHIP_NORMAL=0): the same verdict, and residuals alike to a
thousand times the tolerance."""
import numpy as np
import pytest

from fixedeffects_rocm import api, warmstart

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _problem(seed, K, lost, weights=False):
    """An uneven two-way panel; K columns of noise and effects, and the same with those in `lost` explained in full."""
    rng = np.random.default_rng(seed)
    N, n = 6_007 + 501 * seed, (500 + 30 * seed, 60)
    refs = [rng.integers(1, k + 1, N) for k in n]
    fes = [api.FixedEffect.from_refs(r, k) for r, k in zip(refs, n)]
    fits = [sum(rng.standard_normal(k)[r - 1] for r, k in zip(refs, n)) for _ in range(K)]
    noisy = [f + rng.standard_normal(N) for f in fits]
    some = [f if c in lost else y for c, (f, y) in enumerate(zip(fits, noisy))]
    return fes, rng.lognormal(0, 0.5, N) if weights else None, noisy, some


def _solve(s, Y, start=None):
    cols = [y.copy() for y in Y]
    if start is None:
        _, it, cv = s.solve_residuals_many(cols, tol=TOL, maxiter=1_000)
    else:
        it, cv = warmstart.solve_residuals_from(s, cols, start, tol=TOL, maxiter=1_000)
    return cols, it, cv, [s.lsmr_info(c) for c in range(len(Y))]


def _like_the_passes(got, want, Y, lost):
    for c in lost:
        assert np.linalg.norm(got[0][c] - want[0][c]) <= 1e3 * TOL * np.linalg.norm(Y[c])
        assert got[2][c] == want[2][c]


@pytest.mark.parametrize("algorithm", ["lsmr", "projected"])
@pytest.mark.parametrize("start", [False, True])
@pytest.mark.parametrize("K,lost", [(2, (1,)), (3, (0,)), (5, (0, 3)), (16, (2, 5, 15)), (32, tuple(range(1, 32, 2))),
                                    (32, (31,))])
def test_others_keep_their_results(gpu, monkeypatch, K, lost, start, algorithm):
    fes, w, noisy, some = _problem(1, K, lost, weights=K == 5)
    rng = np.random.default_rng(4)
    x0 = [rng.standard_normal(560 + 30) if c % 3 else None for c in range(K)] if start else None
    with api.FixedEffectSolverROCm(fes, w, "fp64", algorithm=algorithm) as s:
        plain = _solve(s, noisy, x0)
        got = _solve(s, some, x0)
        again = _solve(s, some, x0)
    monkeypatch.setenv("FEHIP_NORMAL", "0")
    with api.FixedEffectSolverROCm(fes, w, "fp64", algorithm=algorithm) as s:
        want = _solve(s, some, x0)
    for c in range(K):
        assert np.array_equal(got[0][c], again[0][c]) and got[3][c] == again[3][c]
        if c not in lost:
            assert np.array_equal(got[0][c], plain[0][c])
            assert (got[1][c], got[2][c], got[3][c]) == (plain[1][c], plain[2][c], plain[3][c])
    _like_the_passes(got, want, some, lost)


@pytest.mark.parametrize("K,lost", [(1, (0,)), (2, (0, 1)), (3, (0, 2)), (32, tuple(range(17)))])
def test_most_columns(gpu, monkeypatch, K, lost):
    fes, w, _, some = _problem(2, K, lost)
    with api.FixedEffectSolverROCm(fes, w) as s:
        got = _solve(s, some)
    monkeypatch.setenv("FEHIP_NORMAL", "0")
    with api.FixedEffectSolverROCm(fes, w) as s:
        want = _solve(s, some)
    _like_the_passes(got, want, some, range(K))


def test_panels(gpu):
    # panels whose columns start over beside panels whose columns do not: as alone
    problems = [_problem(k, K, lost) for k, (K, lost) in enumerate([(1, ()), (4, (1,)), (1, (0,)), (9, (0, 8)), (3, ())])]
    solvers = [api.FixedEffectSolverROCm(fes, w) for fes, w, _, _ in problems]
    alone = [_solve(s, some) for s, (_, _, _, some) in zip(solvers, problems)]
    cols = [[y.copy() for y in some] for _, _, _, some in problems]
    it, cv = api.solve_residuals_panels_host(solvers, cols, tol=TOL, maxiter=1_000)
    for a, c, i, v in zip(alone, cols, it, cv):
        assert all(np.array_equal(x, y) for x, y in zip(a[0], c)) and a[1] == i and a[2] == v
    for s in solvers:
        s.close()
