"""GPU test of scale! (src/SolverCPU.jl:78-89) at the level sizes where its
path changes: bit-exact against the same terms added one after another."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu

# a thread per level up to 128 observations (16 terms at a time), a wave beyond
# (chunks of 1024, 32 terms per turn); 0: a level without observations
SIZES = [0, 1, 2, 15, 16, 17, 127, 128, 129, 143, 160, 161, 1023, 1024, 1025, 1056, 2048, 2049, 5000]


def _sum_in_order(terms, T):
    s = T(0)
    for t in terms:
        s = T(np.float64(s) + t)
    return s


@pytest.mark.parametrize("precision,T", [("fp64", np.float64), ("fp32", np.float32)])
@pytest.mark.parametrize("weights,interacted", [(False, False), (True, False), (False, True), (True, True)])
def test_scale_bits(gpu, precision, T, weights, interacted):
    rng = np.random.default_rng(7)
    refs = rng.permutation(np.repeat(np.arange(1, len(SIZES) + 1), SIZES))
    N = len(refs)
    z = rng.uniform(0.5, 1.5, N) if interacted else None
    w = rng.lognormal(0, 0.5, N) if weights else None
    other = api.FixedEffect.from_refs(rng.integers(1, 31, N), 30)
    with api.FixedEffectSolverROCm([other, api.FixedEffect.from_refs(refs, len(SIZES), z)], w, precision) as s:
        got = s.scale(1)
    for k, size in enumerate(SIZES):
        i = np.flatnonzero(refs == k + 1)
        t = (1.0 if z is None else z[i] * z[i]) * (1.0 if w is None else w[i]) * np.ones(size)
        a = _sum_in_order(t, T)
        want = T(1) / T(np.sqrt(np.float64(a))) if a > 0 else T(0)
        assert got[k] == np.float64(want), (size, got[k], want)
