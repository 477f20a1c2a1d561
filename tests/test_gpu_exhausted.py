"""GPU test of solves whose bidiagonalization ends in rounding: an FE collinear
with the others (in the projected iteration nothing is left to solve for), an
FE given twice, complete grids (exhausted after a step or two), a handful of
levels; columns that the FEs explain in full, or one of them.  Against the
passes over the observations (FEHIP_NORMAL=0): the same verdict, and residuals
alike to 1e-9 of the column, a thousand times the tolerance of the solves."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu


def _refs(shape, rng):
    if shape == "constant":
        return [rng.integers(1, 1_001, 20_011), np.ones(20_011, np.int64)]
    if shape == "constant_large":  # tiles in their own order and in the launches'
        return [rng.integers(1, 60_001, 700_001), np.ones(700_001, np.int64)]
    if shape == "twice":
        r = rng.integers(1, 301, 5_003)
        return [r, rng.integers(1, 41, 5_003), r.copy()]
    if shape == "nested":  # firms inside regions
        r = rng.integers(0, 300, 5_003)
        return [r + 1, r // 30 + 1]
    if shape == "grid":
        a, b, c = np.meshgrid(np.arange(20), np.arange(30), np.arange(7), indexing="ij")
        return [a.ravel() + 1, b.ravel() + 1, c.ravel() + 1]
    if shape == "few":
        return [rng.integers(1, 4, 40), rng.integers(1, 3, 40)]
    return [np.array([1, 2, 2, 3, 3]), np.array([1, 1, 2, 2, 2])]  # "path"


@pytest.mark.parametrize("shape", ["constant", "constant_large", "twice", "nested", "grid", "few", "path"])
@pytest.mark.parametrize("algorithm", ["lsmr", "projected"])
@pytest.mark.parametrize("K", [1, 16])
def test_verdicts(gpu, monkeypatch, shape, algorithm, K):
    rng = np.random.default_rng(5)
    refs = [np.asarray(r, np.int64) for r in _refs(shape, rng)]
    N, n = len(refs[0]), [int(r.max()) for r in refs]
    fit = sum(rng.standard_normal(k)[r - 1] for r, k in zip(refs, n))
    Y = [(rng.standard_normal(N), fit, 1.0 * (refs[0] == 1), np.ones(N))[c % 4] for c in range(max(K, 4))]
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("FEHIP_NORMAL", on)
        with api.FixedEffectSolverROCm([api.FixedEffect.from_refs(r, k) for r, k in zip(refs, n)], None, "fp64",
                                       algorithm=algorithm) as s:
            got = []
            for i in range(0, len(Y), K):
                cols = [y.copy() for y in Y[i:i + K]]
                _, it, cv = s.solve_residuals_many(cols, tol=1e-12, maxiter=1_000)
                got += list(zip(cols, cv, it, [s.lsmr_info(c) for c in range(len(cols))]))
        out[on] = got
    for y, (a, ca, ia, fa), (b, cb, ib, fb) in zip(Y, out["1"], out["0"]):
        print(shape, algorithm, ca, cb, ia, ib, fa["istop"], fb["istop"], np.linalg.norm(a - b) / np.linalg.norm(y))
    for y, (a, ca, ia, fa), (b, cb, ib, fb) in zip(Y, out["1"], out["0"]):
        assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(y)
        assert ca == cb
