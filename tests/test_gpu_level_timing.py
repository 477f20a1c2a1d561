"""GPU test of the timing hooks on handles whose solves iterate in level space:
fehip_time_kernels without weights and for more iterations than a filler LSMR
lasts, and the autotuner's time per iteration, which is that iteration's."""
import ctypes as C

import numpy as np
import pytest

from fixedeffects_rocm import api
from fixedeffects_rocm._lib import check, lib

pytestmark = pytest.mark.gpu


def _times(s, K, reps):
    ms = np.zeros(8)
    check(lib.fehip_time_kernels(s._h, K, reps, ms.ctypes.data_as(C.POINTER(C.c_double))))
    return ms


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("K", [1, 5, 32])
def test_hooks(gpu, K, weights, precision):
    rng = np.random.default_rng(1)
    N, n = 200_003, (20_000, 2_000)
    fes = [api.FixedEffect.from_refs(rng.integers(1, k + 1, N), k) for k in n]
    Y = [rng.standard_normal(N) for _ in range(K)]
    with api.FixedEffectSolverROCm(fes, rng.lognormal(0, 0.5, N) if weights else None, precision) as s:
        for reps in (1, 2, 7, 40):
            ms = _times(s, K, reps)
            assert ms[0] > 0 and ms[1] > 0 and ms[6] > 0 and not ms[2:6].any()
        sched = s.autotune(K=K, reps=3)
        assert sched["ms_per_iter"] == sched["default_ms_per_iter"] > 0  # (no schedule changes it)
        cols = [y.copy() for y in Y]
        _, it, cv = s.solve_residuals_many(cols, tol=1e-10)
        assert all(cv)
