"""GPU tests of solves with little device memory (FEHIP_DEVICE_MB limits what
the library may hold).  Whatever fits without the level-space matrix
(FEHIP_NORMAL=0) fits with it: the matrix is given up, or its vectors, or a
batch of columns that start over, and no call keeps another's scratch."""
import ctypes as C

import numpy as np
import pytest

from fixedeffects_rocm import api, device
from fixedeffects_rocm._lib import FEHIP_EOOM, FehipError

pytestmark = pytest.mark.gpu

N, LEVELS = 300_007, (30_000, 3_000, 9)


def _panel():
    rng = np.random.default_rng(6)
    refs = [rng.integers(1, k + 1, N) for k in LEVELS]
    fes = [api.FixedEffect.from_refs(r, k) for r, k in zip(refs, LEVELS)]
    fit = sum(rng.standard_normal(k)[r - 1] for r, k in zip(refs, LEVELS))
    Y = [fit if c == 3 else fit + rng.standard_normal(N) for c in range(16)]
    return fes, rng.lognormal(0, 0.5, N), Y


def _columns(s, Y, tol=1e-12):
    cols = [y.copy() for y in Y]
    s.solve_residuals_many(cols, tol=tol, maxiter=1_000)
    return cols


def _wider(fes, w, Y, precision):
    # a handle's batches grow and shrink; new weights; coefficients
    with api.FixedEffectSolverROCm(fes, w, precision) as s:
        out = _columns(s, Y[:1]) + _columns(s, Y) + _columns(s, Y[:2])
        s.update_weights(np.sqrt(w))
        out += _columns(s, Y[:2])
        out.append(sum(s.solve_coefficients(Y[0], tol=1e-12)[0]))
        return out + _columns(s, Y)


def _one_batch(fes, w, Y, precision):
    # columns of one batch of which one starts over, again and again
    with api.FixedEffectSolverROCm(fes, w, precision) as s:
        return [c for _ in range(3) for c in _columns(s, Y[:8])]


def _fits(work, *a):
    try:
        return work(*a)
    except FehipError as e:
        assert e.code == FEHIP_EOOM
        return None


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("work", [_wider, _one_batch])
def test_what_fitted_still_fits(gpu, monkeypatch, work, precision):
    fes, w, Y = _panel()
    want = work(fes, w, Y, "fp64")
    monkeypatch.setenv("FEHIP_NORMAL", "0")
    lo, hi = 1, 1_024  # MB: too little, enough
    while hi - lo > 1:
        mid = (lo + hi) // 2
        monkeypatch.setenv("FEHIP_DEVICE_MB", str(mid))
        if _fits(work, fes, w, Y, precision) is None:
            lo = mid
        else:
            hi = mid
    monkeypatch.setenv("FEHIP_NORMAL", "1")
    for limit in sorted({hi + d for d in (0, 1, 2, 3, 5, 8, 13, 21, 34, 55, 89, 144)}):
        monkeypatch.setenv("FEHIP_DEVICE_MB", str(limit))
        got = _fits(work, fes, w, Y, precision)
        assert got is not None, (limit, hi)
        for a, b, y in zip(got, want, Y * 3):
            assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(y), limit


def test_refused_handles_leave_nothing(gpu, monkeypatch):
    fes, w, Y = _panel()
    want = _columns(api.FixedEffectSolverROCm(fes, w), Y[:1])
    for limit in (1, 4, 8):  # MB; the refs and caches alone take more
        monkeypatch.setenv("FEHIP_DEVICE_MB", str(limit))
        assert _fits(api.FixedEffectSolverROCm, fes, w) is None
    monkeypatch.delenv("FEHIP_DEVICE_MB")
    assert np.array_equal(_columns(api.FixedEffectSolverROCm(fes, w), Y[:1])[0], want[0])


def test_trim(gpu):
    hip = device._hip
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    fes, w, Y = _panel()
    _one_batch(fes, w, Y, "fp64")
    kept = free()
    api.trim()
    assert free() - kept >= 8 * N * 8  # at least one batch's columns
    _one_batch(fes, w, Y, "fp64")
