"""GPU test of matrices with enough tiles that those inside long rows are
visited by column (csrc/normal.hip, tile_order): long rows before and after the
FE of most levels, one alone, none; against the passes over the observations
(FEHIP_NORMAL=0).  tol 1e-12 determines the residual to about 1e-10; the bar is
ten times that."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [(60_000, 4_000, 12), (11, 60_000, 3), (60_000, 1), (60_000, 5_000)])
@pytest.mark.parametrize("algorithm", ["lsmr", "projected"])
@pytest.mark.parametrize("K", [1, 3])
def test_orders(gpu, monkeypatch, levels, algorithm, K):
    rng = np.random.default_rng(sum(levels))
    N = 700_001  # over a million entries: more than 2048 tiles (one 60000-entry row and its column: fewer)
    fes = [api.FixedEffect.from_refs(rng.integers(1, k + 1, N), k) for k in levels]
    Y = [rng.standard_normal(N) for _ in range(K)]
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("FEHIP_NORMAL", on)
        cols = [y.copy() for y in Y]
        with api.FixedEffectSolverROCm(fes, None, "fp64", algorithm=algorithm) as s:
            _, it, cv = s.solve_residuals_many(cols, tol=1e-12, maxiter=10_000)
        out[on] = cols, it, cv
    assert out["1"][2] == out["0"][2]
    for a, b in zip(out["1"][0], out["0"][0]):
        assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
    assert all(abs(i - j) <= 2 for i, j in zip(out["1"][1], out["0"][1]))
