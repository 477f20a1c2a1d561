"""GPU test of the rule that leaves narrow batches to the passes over the
observations where most of the matrix's entries gather from large vectors: three
FEs of more than 2^18 levels (csrc/fehip.hip, takes_level), narrow and wide
batches in either order, against FEHIP_NORMAL=0.  tol 1e-12 determines the
residual to about 1e-10; the bar is ten times that."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order", [(1, 8, 2), (8, 1)])
def test_widths_in_turn(gpu, monkeypatch, order, precision):
    rng = np.random.default_rng(3)
    N, n = 1_500_007, (300_000, 280_000, 270_000)
    fes = [api.FixedEffect.from_refs(rng.integers(1, k + 1, N), k) for k in n]
    Y = [rng.standard_normal(N) for _ in range(max(order))]
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("FEHIP_NORMAL", on)
        with api.FixedEffectSolverROCm(fes, None, precision if on == "1" else "fp64") as s:
            got = []
            for K in order:
                cols = [y.copy() for y in Y[:K]]
                _, it, cv = s.solve_residuals_many(cols, tol=1e-12, maxiter=2_000)
                got.append((cols, it, cv))
                if K < 8 and precision == "fp64":
                    # a narrow batch is the passes' in both, bit for bit
                    out.setdefault(("narrow", on), []).append(cols)
        out[on] = got
    for (a, ia, ca), (b, ib, cb) in zip(out["1"], out["0"]):
        assert ca == cb and all(ca)
        for x, y in zip(a, b):
            assert np.linalg.norm(x - y) <= 1e-9 * np.linalg.norm(y)
    for a, b in zip(out.get(("narrow", "1"), []), out.get(("narrow", "0"), [])):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
