"""GPU tests of the memory a handle takes and gives back (csrc/hostmem.h):
blocks reused by later handles and by handles of other threads hold no trace
of the work before, and copies of the caller's memory are whole at the sizes
where their path changes."""
import threading

import numpy as np
import pytest

from fixedeffects_rocm import api, synth
from fixedeffects_rocm._lib import FEHIP_EREF, FehipError

pytestmark = pytest.mark.gpu


def _panel(seed):
    # sizes differ by seed, so later handles get blocks of other shapes
    return synth.worker_firm(20_000 + 3_777 * seed, 2_000 + 300 * seed, 200 + 17 * seed, 12, 0.05, 1.1, 2, seed=seed)


def _solve(p):
    fes = [api.FixedEffect.from_refs(r, n, z) for r, n, z in zip(p.refs, p.n, p.interactions)]
    with api.FixedEffectSolverROCm(fes, p.weights) as s:
        cols = [p.Y[:, k].copy() for k in range(p.K)]
        _, it, cv = s.solve_residuals_many(cols, tol=1e-10, maxiter=1000)
    return cols, it, cv


def _same(a, b):
    return a[1:] == b[1:] and all(np.array_equal(x, y) for x, y in zip(a[0], b[0]))


def test_reused_blocks_change_nothing(gpu):
    # each panel on blocks that the others used, twice: bitwise the same
    panels = [_panel(k) for k in range(4)]
    first = [_solve(p) for p in panels]
    again = [_solve(p) for p in reversed(panels)][::-1]
    assert all(_same(a, b) for a, b in zip(first, again))


def test_handles_of_several_threads(gpu):
    panels = [_panel(k) for k in range(4)]
    want = [_solve(p) for p in panels]
    got = [[None] * 3 for _ in panels]

    def work(k):
        for i in range(3):
            got[k][i] = _solve(panels[k])

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(panels))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(r is not None and _same(r, w) for g, w in zip(got, want) for r in g)


# the copies take the runtime's path or the staged one: 2 MB from the device,
# 32 MB to it (8-byte elements), and remainders of a chunk
@pytest.mark.parametrize("N", [262_143, 262_145, 4_194_303, 4_194_305, 5_000_011])
def test_grouping_copies(gpu, N):
    rng = np.random.default_rng(N)
    keys = rng.integers(-50, 1_000, N) * 3
    refs, n = api.group(keys)
    u, inv = np.unique(keys, return_inverse=True)
    assert n == len(u) and np.array_equal(refs, inv + 1)


@pytest.mark.parametrize("N", [4_194_303, 4_194_305, 4_500_007])
def test_refs_narrowed_on_the_way(gpu, N):
    rng = np.random.default_rng(N)
    a, b = rng.integers(1, 301, N), rng.integers(1, 41, N)
    fes = [api.FixedEffect.from_refs(a, 300), api.FixedEffect.from_refs(b, 40)]
    with api.FixedEffectSolverROCm(fes) as s:
        perm, off = s.csr(1)
    assert np.array_equal(perm, np.argsort(b, kind="stable"))
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(np.bincount(b - 1, minlength=40))]))
    for bad in (0, 41, 1 << 32, -(1 << 32) + 5):
        b[N - 3] = bad
        with pytest.raises(FehipError) as e:
            api.FixedEffectSolverROCm([api.FixedEffect.from_refs(a, 300), api.FixedEffect.from_refs(b, 40)])
        assert e.value.code == FEHIP_EREF


@pytest.mark.parametrize("bad", [0.0, -1.0, np.inf, np.nan])
def test_refused_weights_leave_the_handle(gpu, bad):
    p = _panel(1)
    fes = [api.FixedEffect.from_refs(r, n) for r, n in zip(p.refs, p.n)]
    with api.FixedEffectSolverROCm(fes, p.weights) as s:
        want = s.solve_residuals(p.Y[:, 0].copy(), tol=1e-10)
        w = p.weights.copy()
        w[[17, 1_234]] = bad
        with pytest.raises(FehipError, match="observation 18"):
            s.update_weights(w)
        got = s.solve_residuals(p.Y[:, 0].copy(), tol=1e-10)
    assert np.array_equal(got[0], want[0]) and got[1:] == want[1:]
