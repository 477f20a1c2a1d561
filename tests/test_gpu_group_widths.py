"""GPU grouping of several columns at the widths where its path changes: the
ranges of all columns in one 64-bit word, or each column numbered alone.
Integer work, so bit-exact against numpy's unique on the host."""
import numpy as np
import pytest

from fixedeffects_rocm import api

pytestmark = pytest.mark.gpu


def _column(rng, N, bits):
    # a column whose range needs exactly `bits` bits, with ties
    if bits == 0:
        return np.full(N, -7, np.int64)
    pool = rng.integers(0, 2 ** 64 - 1, 40, dtype=np.uint64, endpoint=True) >> np.uint64(64 - bits)
    pool[:2] = 0, 2 ** bits - 1
    return (rng.permutation(np.concatenate([pool[:2], rng.choice(pool, N - 2)])) + np.uint64(2 ** 63)).view(np.int64)


@pytest.mark.parametrize("widths", [(0, 0), (0, 5, 0), (8, 8), (64, 0), (0, 64), (31, 33), (33, 32), (1, 62, 1),
                                    (21, 21, 22, 1), (63, 1), (64, 1)])
def test_widths(gpu, widths):
    rng = np.random.default_rng(sum(widths))
    cols = [_column(rng, 4_099, b) for b in widths]
    refs, n = api.group(*cols)
    want = api.FixedEffect(*cols)
    assert n == want.n
    np.testing.assert_array_equal(refs, want.refs)
