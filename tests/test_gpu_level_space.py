"""GPU tests of the level-space iteration (csrc/normal.hip) against the passes
over the observations (FEHIP_NORMAL=0) on the forms both accept: FE counts,
orders of the FEs, interactions, weights, levels without observations, rows
from empty to many tiles long, every batch width, the projected algorithm and
the precisions that use it.

Both sides solve to tol 1e-12, where the residual is determined to about 1e-10
by the data (tests/test_gpu_parity.py); the bar is ten times that."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu

RTOL = 1e-9


def _fe(rng, N, n, interacted=False, gaps=0, giant=0.0):
    """Refs of one FE: uniform over n levels, `gaps` more levels without
    observations spread among them, a share `giant` of them in one level."""
    r = rng.integers(0, n, N)
    if giant:
        r[rng.random(N) < giant] = n // 2
    ids = np.sort(rng.choice(n + gaps, n, replace=False)) + 1
    return api.FixedEffect.from_refs(ids[r], n + gaps, rng.uniform(0.5, 1.5, N) if interacted else None)


def _solve(monkeypatch, on, fes, w, Y, precision="fp64", algorithm="lsmr"):
    monkeypatch.setenv("FEHIP_NORMAL", "1" if on else "0")
    cols = [y.copy() for y in Y]
    with api.FixedEffectSolverROCm(fes, w, precision, algorithm=algorithm) as s:
        _, it, cv = s.solve_residuals_many(cols, tol=1e-12, maxiter=20_000)
        assert all(cv)
        again = [y.copy() for y in Y]
        s.solve_residuals_many(again, tol=1e-12, maxiter=20_000)
    assert all(np.array_equal(a, b) for a, b in zip(cols, again))  # bitwise repeatable
    return cols, it


def _compare(monkeypatch, fes, w, Y, **kw):
    a, ia = _solve(monkeypatch, True, fes, w, Y, **kw)
    b, ib = _solve(monkeypatch, False, fes, w, Y, **kw)
    for x, y, z in zip(a, b, Y):
        # (relative to the column where the fixed effects explain all of it)
        assert np.linalg.norm(x - y) <= RTOL * max(np.linalg.norm(y), 1e-3 * np.linalg.norm(z))
    if kw.get("precision") != "mixed":  # the mixed mode's two phases count differently
        assert all(abs(i - j) <= 2 for i, j in zip(ia, ib))


@pytest.mark.parametrize("K", [1, 2, 3, 8, 16, 32])
@pytest.mark.parametrize("shape", ["giant_row", "gaps", "few_levels_first"])
def test_shapes(gpu, monkeypatch, shape, K):
    rng = np.random.default_rng(K)
    N = 20_011
    if shape == "giant_row":  # one level of half the observations: its row spans many tiles
        fes = [_fe(rng, N, 3_000, giant=0.5), _fe(rng, N, 700), _fe(rng, N, 9)]
    elif shape == "gaps":  # empty rows between the others, whole tiles of them
        fes = [_fe(rng, N, 900, gaps=5_000), _fe(rng, N, 300, gaps=40), _fe(rng, N, 70, gaps=1)]
    else:  # FE s last, a few-level FE before it
        fes = [_fe(rng, N, 12), _fe(rng, N, 200), _fe(rng, N, 2_500)]
    w = rng.lognormal(0, 0.5, N) if K != 2 else None
    _compare(monkeypatch, fes, w, [rng.standard_normal(N) for _ in range(K)])


@pytest.mark.parametrize("N", [2, 5, 63, 65, 257, 1_031])
def test_small(gpu, monkeypatch, N):
    rng = np.random.default_rng(N)
    fes = [_fe(rng, N, max(1, N // 3)), _fe(rng, N, max(1, N // 7))]
    _compare(monkeypatch, fes, None, [rng.standard_normal(N)])


@pytest.mark.parametrize("algorithm", ["lsmr", "projected"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("inter", [(), (0,), (2,), (0, 1, 2, 3)])
def test_forms(gpu, monkeypatch, inter, precision, algorithm):
    rng = np.random.default_rng(len(inter) + 10)
    N = 9_973
    fes = [_fe(rng, N, n, interacted=g in inter, giant=0.2 * (g == 1)) for g, n in enumerate((40, 1_200, 300, 7))]
    _compare(monkeypatch, fes, rng.lognormal(0, 0.5, N), [rng.standard_normal(N) for _ in range(5)],
             precision=precision, algorithm=algorithm)


def test_new_weights(gpu, monkeypatch):
    # the matrix follows update_weights, also to unit weights and back
    rng = np.random.default_rng(3)
    N = 30_011
    fes = [_fe(rng, N, 2_000, giant=0.1), _fe(rng, N, 300), _fe(rng, N, 11)]
    ws = [None, rng.lognormal(0, 0.5, N), None, rng.lognormal(0, 1.0, N)]
    y = rng.standard_normal(N)
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("FEHIP_NORMAL", on)
        with api.FixedEffectSolverROCm(fes, ws[1]) as s:
            out[on] = [s.update_weights(w).solve_residuals(y.copy(), tol=1e-12)[0] for w in ws]
    for a, b in zip(out["1"], out["0"]):
        assert np.linalg.norm(a - b) <= RTOL * np.linalg.norm(b)


def test_many_entries_keep_the_observation_passes(gpu, monkeypatch):
    # nine FEs: more entries than the passes over the observations read
    rng = np.random.default_rng(9)
    N = 4_001
    fes = [_fe(rng, N, n) for n in (300, 200, 150, 120, 100, 90, 80, 70, 66)]
    _compare(monkeypatch, fes, None, [rng.standard_normal(N)])
