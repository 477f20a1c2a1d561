"""GPU test of scale! (src/SolverCPU.jl:78-89) at the sizes where a large
level's kernel turns from one chunk of 1536 terms to the next (two buffers in
turn, 32 terms a step, read ahead past a chunk's end): bit-exact against the
same terms added one after another."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu

SIZES = [c + d for c in (1536, 3072, 4608) for d in (-33, -1, 0, 1, 31, 32)]


@pytest.mark.parametrize("precision,T", [("fp64", np.float64), ("fp32", np.float32)])
@pytest.mark.parametrize("weights,interacted", [(True, False), (False, True), (True, True)])
def test_chunk_ends(gpu, precision, T, weights, interacted):
    rng = np.random.default_rng(17)
    refs = rng.permutation(np.repeat(np.arange(1, len(SIZES) + 1), SIZES))
    N = len(refs)
    z = rng.uniform(0.5, 1.5, N) if interacted else None
    w = rng.lognormal(0, 0.5, N) if weights else None
    other = api.FixedEffect.from_refs(rng.integers(1, 31, N), 30)
    with api.FixedEffectSolverROCm([other, api.FixedEffect.from_refs(refs, len(SIZES), z)], w, precision) as s:
        got = s.scale(1)
    for k, size in enumerate(SIZES):
        i = np.flatnonzero(refs == k + 1)
        a = T(0)
        for t in (1.0 if z is None else z[i] * z[i]) * (1.0 if w is None else w[i]) * np.ones(size):
            a = T(np.float64(a) + t)
        assert got[k] == np.float64(T(1) / T(np.sqrt(np.float64(a)))), size
