"""GPU tests of the memory a handle takes and gives back (csrc/hostmem.h):
blocks reused by later handles and by handles of other threads hold no trace
of the work before, and copies of the caller's memory are whole at the sizes
where their path changes."""
import threading

import numpy as np
import pytest

from fixedeffects_rocm import api, synth

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
