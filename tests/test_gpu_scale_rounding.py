"""GPU test of level space where scale!'s serial sums are off by many eps: a
million equal weights of 0.1 in a level (1.3e-11), random weights, a constant
FE that the others explain, large levels in the FE that the projected iteration
eliminates.  Against the passes over the observations (FEHIP_NORMAL=0): the
same verdict, and residuals alike to a thousand times the tolerance."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu


def _refs(shape, rng):
    N = 1_200_007
    if shape == "constant":  # one level of all observations
        return [rng.integers(1, 60_001, N), np.ones(N, np.int64)], 1e-12
    if shape == "constant_s_large":  # the eliminated FE's levels hold 6000 each
        return [rng.integers(1, 201, N), np.ones(N, np.int64)], 1e-10
    if shape == "few":  # 30000 and 40000 observations a level
        return [rng.integers(1, 31, N), rng.integers(1, 41, N)], 1e-10
    return [rng.integers(1, 100_001, N), rng.integers(1, 5_001, N), rng.integers(1, 4, N)], 1e-12  # "three"


@pytest.mark.parametrize("shape", ["constant", "constant_s_large", "few", "three"])
@pytest.mark.parametrize("weights", ["tenth", "random", "mixed"])
@pytest.mark.parametrize("algorithm", ["lsmr", "projected"])
@pytest.mark.parametrize("K", [1, 16])
def test_verdicts(gpu, monkeypatch, shape, weights, algorithm, K):
    rng = np.random.default_rng(8)
    refs, tol = _refs(shape, rng)
    N, n = len(refs[0]), [int(r.max()) for r in refs]
    w = {"tenth": np.full(N, 0.1), "random": rng.lognormal(0, 0.5, N),
         "mixed": np.where(rng.random(N) < 0.5, 0.1, 0.7)}[weights]
    fit = sum(rng.standard_normal(k)[r - 1] for r, k in zip(refs, n))
    Y = [(rng.standard_normal(N), fit, 1.0 * (refs[0] == 1), np.ones(N))[c % 4] for c in range(max(K, 4))]
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("FEHIP_NORMAL", on)
        got = []
        with api.FixedEffectSolverROCm([api.FixedEffect.from_refs(r, k) for r, k in zip(refs, n)], w, "fp64",
                                       algorithm=algorithm) as s:
            for i in range(0, len(Y), K):
                cols = [y.copy() for y in Y[i:i + K]]
                _, it, cv = s.solve_residuals_many(cols, tol=tol, maxiter=500)
                got += list(zip(cols, cv, it, [s.lsmr_info(c) for c in range(len(cols))]))
        out[on] = got
    for y, (a, ca, ia, fa), (b, cb, ib, fb) in zip(Y, out["1"], out["0"]):
        print(shape, weights, algorithm, ca, cb, ia, ib, fa["istop"], fb["istop"],
              np.linalg.norm(a - b) / np.linalg.norm(y))
    for y, (a, ca, ia, fa), (b, cb, ib, fb) in zip(Y, out["1"], out["0"]):
        assert np.linalg.norm(a - b) <= 1e3 * tol * np.linalg.norm(y)
        assert ca == cb


def test_algorithms_in_turn(gpu):
    # the matrix's values differ between the two iterations where the eliminated FE has large levels
    rng = np.random.default_rng(2)
    N = 300_007
    refs = [rng.integers(1, 61, N), rng.integers(1, 41, N), rng.integers(1, 8, N)]
    fes = [api.FixedEffect.from_refs(r, int(r.max())) for r in refs]
    w, y = np.full(N, 0.1), rng.standard_normal(N)
    want = {}
    for a in ("lsmr", "projected"):
        with api.FixedEffectSolverROCm(fes, w, "fp64", algorithm=a) as s:
            want[a] = s.solve_residuals(y.copy(), tol=1e-10)
    with api.FixedEffectSolverROCm(fes, w, "fp64") as s:
        for a in ("projected", "lsmr", "projected", "lsmr"):
            got = s.set_algorithm(a).solve_residuals(y.copy(), tol=1e-10)
            assert np.array_equal(got[0], want[a][0]) and got[1:] == want[a][1:]
            s.update_weights(w)
