"""GPU normalize! where components change hands: one workgroup up to 16384
levels, 128 of them beyond.  Sums in another order than the oracle's; a mean of
L unit-size values differs by about sqrt(L) eps at most: 1e-12."""
import numpy as np
import pytest

import oracle
from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(16384,), (16385,), (16383, 16386, 5), (40_000, 2, 17_000, 17_000, 300)])
@pytest.mark.parametrize("G", [2, 3])
def test_sizes(gpu, sizes, G):
    # component k: sizes[k] levels, one in the last FE and in the one before
    # (three FEs), the others in the first, linked by one observation each
    rng = np.random.default_rng(sum(sizes) + G)
    first = [np.full(s - (G - 1), k) for k, s in enumerate(sizes)]
    block = np.concatenate(first)
    perm = rng.permutation(len(block))
    refs = [np.arange(1, len(block) + 1)[perm]] + [block[perm] + 1 for _ in range(G - 1)]
    n = [len(block) + 2] + [len(sizes)] * (G - 1)
    coefs = [rng.standard_normal(k) for k in n]
    want = oracle.normalize([c.copy() for c in coefs], refs, n, [True] * G)
    fes = [api.FixedEffect.from_refs(r, k) for r, k in zip(refs, n)]
    with api.FixedEffectSolverROCm(fes, None, "fp64") as s:
        got = s.normalize([c.copy() for c in coefs])
        again = s.normalize([c.copy() for c in coefs])
    for a, b, c in zip(got, want, again):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-12)
        np.testing.assert_array_equal(a, c)
