"""CPU tests of the level-space form of the LSMR iteration (csrc/normal.hip):
its recurrences against LSMR on the observations, and the cutting of the
normal matrix's entries into tiles, both restated in numpy."""
import numpy as np
import pytest
import scipy.sparse as sp

from fixedeffects_rocm import synth

# csrc/normal.h
TILE, SLACK, ROW = 512, 128, 8
CAP, ROWS = TILE + SLACK, (TILE + SLACK) // ROW + 2


def _map(p):
    """The scaled fixed-effect map with the weights' square roots, and those."""
    sw = np.sqrt(p.weights)
    blocks = []
    for r, n, z in zip(p.refs, p.n, p.interactions):
        z = np.ones(p.N) if z is None else z
        s2 = np.bincount(r - 1, p.weights * z * z, n)
        sc = np.where(s2 > 0, 1 / np.sqrt(np.where(s2 > 0, s2, 1)), 0)
        blocks.append(sp.csr_matrix((sw * z * sc[r - 1], (np.arange(p.N), r - 1)), shape=(p.N, n)))
    return sp.hstack(blocks).tocsr(), sw


def _iterate(A, b, k, level_space):
    """k bidiagonalization steps from x0 = A'b: alpha and beta of each (src/utils/lsmr.jl:63-68, :104-110)."""
    At = A.T.tocsr()
    M = (At @ A).tocsr()
    u = b - A @ (At @ b)
    beta = np.linalg.norm(u)
    u /= beta
    v = At @ u
    alpha = np.linalg.norm(v)
    v /= alpha
    out, old = [], np.zeros_like(v)
    for i in range(k):
        if level_space:
            q = M @ v
            a = v @ q
            g = 0.0 if i == 0 else alpha * beta
            w = q - a * v - g * old
            beta = np.sqrt(max(a - alpha * alpha, 0.0))
            nw = np.linalg.norm(w)
            old, v, alpha = v, w / nw, nw / beta
        else:
            u = A @ v - alpha * u
            beta = np.linalg.norm(u)
            u /= beta
            v = At @ u - beta * v
            alpha = np.linalg.norm(v)
            v /= alpha
        out.append((alpha, beta))
    return np.array(out)


@pytest.mark.parametrize("name,scale", [("worker_firm_1e7", 0.002), ("worker_firm_1e8_k16", 0.0002)])
def test_recurrences(name, scale):
    # the same alpha and beta to rounding while Lanczos is in its first dozen
    # steps (later ones part for any order of sums, see test_oracle.py)
    p = synth.config(name, scale=scale)
    A, sw = _map(p)
    b = sw * p.Y[:, 0]
    np.testing.assert_allclose(_iterate(A, b, 12, True), _iterate(A, b, 12, False), rtol=1e-12)


def _tiles(off, ra, rb, T, slack=SLACK):
    """k_nf_tiles: (first entry, first row, row cut by the start or -1) per tile."""
    f = off[ra:rb + 1] - off[ra] + ROW * np.arange(rb - ra + 1)
    out = []
    for k in range(-(-int(f[-1]) // T)):
        u = k * T
        lo = ra + int(np.searchsorted(f, u, side="left"))
        r, e, cut = lo, int(off[lo]), -1
        if lo > ra and f[lo - ra] - u > slack:
            inside = u - int(f[lo - 1 - ra]) - ROW
            if inside > 0:
                e, cut = int(off[lo - 1]) + inside, lo - 1
            else:
                r, e = lo - 1, int(off[lo - 1])
        out.append((e, r, cut))
    return out


def _check(off, T, slack=SLACK):
    p = len(off) - 1
    t = _tiles(off, 0, p, T, slack)
    e = np.array([x[0] for x in t] + [off[-1]])
    r = np.array([x[1] for x in t] + [p])
    assert (np.diff(e) >= 0).all() and (np.diff(r) >= 0).all() and e[0] == 0 and r[0] == 0
    assert np.diff(e).max() <= CAP and np.diff(r).max() < ROWS
    # each row from its owner's part and the head parts of the tiles after it
    val = np.arange(1, off[-1] + 1)
    got = np.zeros(p, np.int64)
    for k in range(len(t)):
        for row in range(r[k], r[k + 1]):
            assert off[row] >= e[k]
            got[row] += val[off[row]:min(off[row + 1], e[k + 1])].sum()
        first = min(off[r[k]], e[k + 1])
        if first > e[k]:
            assert t[k][2] == r[k] - 1 and off[r[k] - 1] < e[k] < off[r[k]]
            got[r[k] - 1] += val[e[k]:first].sum()
        else:
            assert t[k][2] == -1 or off[t[k][2] + 1] == off[t[k][2]]
    want = np.add.reduceat(np.append(val, 0), np.minimum(off[:-1], off[-1])) * (np.diff(off) > 0)
    return np.array_equal(got, want)


@pytest.mark.parametrize("T", [128, 129, 500, 512])
def test_tiles_cover_rows(T):
    rng = np.random.default_rng(T)
    shapes = [rng.integers(0, 6, 4000), np.full(3, 700), np.array([5000]), np.zeros(1000, int),
              np.concatenate([rng.integers(0, 4, 500), [0, 0, 3000, 0, 129, 128, 127, 0], rng.integers(100, 700, 40)]),
              np.concatenate([np.zeros(300, int), [513], np.zeros(300, int), [1]]), np.array([1])]
    for lens in shapes:
        assert _check(np.concatenate([[0], np.cumsum(lens)]), T)
