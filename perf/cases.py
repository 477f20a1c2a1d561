"""Workloads the framework's speed is measured on.

Each case is one call (or one step of a loop) a program makes through the
public API: a resident handle solved again and again, the one-call form that
builds and drops its handle, a reweighting step, batched columns, the mixed
and projected modes, coefficients, key grouping and many panels at once.

The panels are those of ``fixedeffects_rocm.synth`` (uniform two-way, and
Zipf-sized workers moving between firms over years) plus a worker-firm network
whose firms neighbour each other, drawn on the GPU with torch.

Two programs' sums of the same residual in another order stop LSMR one
iteration apart when its tolerance is loose (1e-8 leaves the residual at
about 1e-6), so the FP64 cases ask for a tolerance at which the residual is
determined by its inputs.

torch and libfehip share one process here, so they have to share one HIP
runtime: torch's is made visible to libfehip before libfehip is loaded.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "fixedeffects.jl_amd"))
_runtime = os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so")
if os.path.exists(_runtime):
    ctypes.CDLL(_runtime, mode=ctypes.RTLD_GLOBAL)

from fixedeffects_rocm import api  # noqa: E402

TOL64 = 1e-13   # FP64 and mixed: the residual no longer depends on the order of sums
TOL32 = 1e-6    # Float32 mode: the API's default
MAXITER = 10_000
DEV = "cuda"


def _case(name=None, **over):
    c = dict(kind="resident", shape="worker_firm", N=1000, n1=100, n2=10, n3=0, mobility=0.05, K=1,
             precision="fp64", algorithm="lsmr", weights=False, interacted=False, panels=1)
    c.update(over)
    if name is not None:
        c = {"name": name, **c}
    return c


def listed():
    return [
        # a small estimation solved over and over on a kept handle (a bootstrap, a Newton loop): latency
        _case("small_resident", kind="host", shape="two_way", N=10_000, n1=1_000, n2=50),
        # one call on a small data set, handle and all: the reference's CPU configuration
        _case("one_call_1e5", kind="call", shape="two_way", N=100_000, n1=10_000, n2=100),
        # one step of an iteratively reweighted fit (a Poisson regression): new weights, outcome and regressors
        _case("reweighted_1e6", kind="reweight", N=1_000_003, n1=100_000, n2=10_000, n3=20, K=4, weights=True),
        # the headline drop-in: one column of a worker/firm/year panel, columns resident on the device
        _case("drop_in_1e7", N=10_000_000, n1=1_000_000, n2=100_000, n3=20, weights=True),
        # a regression's 32 variables on that panel in one batch
        _case("batch32_1e7", N=10_000_000, n1=1_000_000, n2=100_000, n3=20, K=32, weights=True),
        # the mixed mode on the interacted panel (years x z), 16 columns
        _case("mixed16_interacted_2e7", N=20_000_000, n1=1_000_000, n2=100_000, n3=50, mobility=0.02, K=16,
              precision="mixed", weights=True, interacted=True),
        # the projected LSMR, a few columns, ragged sizes, no weights
        _case("projected8_ragged", N=6_543_217, n1=654_321, n2=65_431, n3=13, K=8, algorithm="projected"),
        # one call on a large, well-conditioned two-way problem: reading the data and setting up weigh most
        _case("one_call_1e7", kind="call", shape="two_way", N=10_000_000, n1=100_000, n2=100),
        # the API's default call, Float32, on a worker-firm network of neighbouring firms
        _case("float32_network_8e5", kind="call", shape="network", N=800_000, n1=100_000, n2=12_500,
              precision="fp32"),
        # the fixed effects themselves: solve, normalize, one value per observation
        _case("coefficients_2e6", kind="coefficients", shape="two_way", N=2_000_000, n1=200_000, n2=20_000),
        # a fixed effect from two raw key columns (worker x firm), numbered on the device
        _case("group_1e7", kind="group", N=10_000_000, n1=1_000_000, n2=100_000),
        # many regions or industries at once, each its own panel of uneven size
        _case("panels_24", kind="panels", N=400_000, n3=20, K=4, panels=24, weights=True),
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["host", "call", "reweight", "resident", "resident", "resident", "call32", "coefficients",
                       "group", "panels"])
    if kind == "host":
        N = _log(rng, 5_000, 400_000)
        return _case(kind="host", shape=rng.choice(["two_way", "worker_firm"]), N=N, n1=max(50, N // rng.randint(8, 14)),
                     n2=rng.randint(20, 300), K=rng.choice([1, 1, 2, 3, 7]), weights=rng.random() < 0.5)
    if kind == "call":
        N = _log(rng, 50_000, 10_000_000)
        return _case(kind="call", shape="two_way", N=N, n1=max(100, N // rng.randint(20, 200)),
                     n2=rng.choice([12, 60, 100, 500, 2_000]), K=rng.choice([1, 1, 3]), weights=rng.random() < 0.5)
    if kind == "call32":
        N = _log(rng, 200_000, 2_000_000)
        return _case(kind="call", shape="network", N=N, n1=N // 8, n2=N // 64, precision="fp32")
    if kind == "reweight":
        N = _log(rng, 200_000, 3_000_000)
        return _case(kind="reweight", N=N, n1=N // rng.randint(8, 15), n2=N // rng.randint(80, 150),
                     n3=rng.choice([0, 7, 20]), K=rng.randint(1, 5), weights=True)
    if kind == "resident":
        K = rng.choice([1, 2, 5, 8, 16, 20, 32])
        N = _log(rng, 500_000, min(20_000_000, 240_000_000 // K))
        return _case(N=N, n1=N // rng.randint(8, 20), n2=N // rng.randint(80, 200), n3=rng.choice([0, 5, 20, 50]),
                     mobility=rng.choice([0.03, 0.05, 0.1]), K=K, precision=rng.choice(["fp64", "fp64", "mixed"]),
                     algorithm=rng.choice(["lsmr", "lsmr", "projected"]), weights=rng.random() < 0.6)
    if kind == "coefficients":
        N = _log(rng, 100_000, 4_000_000)
        return _case(kind="coefficients", shape="two_way", N=N, n1=N // rng.randint(8, 20), n2=N // rng.randint(80, 200),
                     weights=rng.random() < 0.5)
    if kind == "group":
        N = _log(rng, 200_000, 12_000_000)
        return _case(kind="group", N=N, n1=N // rng.randint(4, 30), n2=N // rng.randint(50, 300))
    return _case(kind="panels", N=_log(rng, 100_000, 500_000), n3=rng.choice([0, 20]), K=rng.randint(1, 5),
                 panels=rng.randint(6, 24), weights=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# panels
# ---------------------------------------------------------------------------
def _zipf_sizes(N, n, s=1.1, least=2):
    """max(least, floor(C k^-s)), k = 1..n, with C found by bisection so that they sum to about N; the rest goes to the first."""
    kp = torch.arange(1, n + 1, dtype=torch.float64, device=DEV) ** (-s)
    lo, hi = 0.0, float(N)
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        if int(torch.clamp(torch.floor(mid * kp), min=least).sum()) <= N:
            lo = mid
        else:
            hi = mid
    sizes = torch.clamp(torch.floor(lo * kp), min=least).to(torch.int64)
    sizes[0] += N - int(sizes.sum())
    return sizes


def _dense(ids):
    """0-based ids without gaps, and how many there are."""
    present = torch.bincount(ids) > 0
    return (torch.cumsum(present, 0) - 1)[ids], int(present.sum())


def _panel(c, seed, K=None):
    """One panel on the GPU: 0-based refs and level counts, interactions, weights (or None) and Y (K x N, float64)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    N, n1, n2, K = c["N"], c["n1"], c["n2"], c["K"] if K is None else K

    def ints(n, size):
        return torch.randint(0, n, (size,), generator=g, device=DEV)

    def normal(*size):
        return torch.randn(*size, generator=g, device=DEV, dtype=torch.float64)

    if c["shape"] == "worker_firm":
        n1 = min(n1, N // 2)
        sizes = _zipf_sizes(N, n1)
        first = torch.zeros(N, dtype=torch.bool, device=DEV)
        first[torch.cumsum(sizes, 0) - sizes] = True
        move = first | (torch.rand(N, generator=g, device=DEV) < c["mobility"])
        worker = torch.repeat_interleave(torch.arange(n1, device=DEV), sizes)
        spell = torch.cumsum(move, 0) - 1
        firm = ints(n2, int(spell[-1]) + 1)[spell]
        order = torch.randperm(N, generator=g, device=DEV)
        ids = [worker[order], firm[order]]
    elif c["shape"] == "network":
        worker = ints(n1, N)
        firm = torch.clamp(worker * n2 // n1 + torch.randint(-40, 41, (N,), generator=g, device=DEV), 0, n2 - 1)
        ids = [worker, firm]
    else:
        ids = [ints(n1, N), ints(n2, N)]
    if c["n3"]:
        ids.append(ints(c["n3"], N))
    refs, n = zip(*(_dense(i) for i in ids))
    effects = [normal(k) for k in n]
    z = [None] * len(refs)
    if c["interacted"]:
        z[-1] = torch.rand(N, generator=g, device=DEV, dtype=torch.float64) + 0.5
    Y = normal(K, N)
    for k in range(K):  # the outcome, then regressors that share less of the effects
        for e, r, m in zip(effects, refs, (1.0, 1.0, 1.0) if k == 0 else (0.5, 0.3, 0.0)):
            if m:
                Y[k] += m * e[r]
    w = torch.exp(0.5 * normal(N)) if c["weights"] else None
    return {"refs": list(refs), "n": list(n), "z": z, "w": w, "Y": Y}


def _fes(p):
    return [api.FixedEffect.from_refs((r + 1).cpu().numpy(), n, None if z is None else z.cpu().numpy())
            for r, n, z in zip(p["refs"], p["n"], p["z"])]


def _host(t):
    return None if t is None else t.cpu().numpy()


def _sizes(c):
    """(N, K) of each panel of one call: sizes log-uniform over a factor of 40 up to N, 1..K columns each."""
    return [(int(c["N"] * 40 ** -((0.618034 * i) % 1.0)), 1 + 7 * i % c["K"]) for i in range(c["panels"])]


def _uneven(c, seed):
    rng = np.random.default_rng(int(seed))
    out = []
    for i, (N, K) in enumerate(_sizes(c)):
        sub = dict(c, N=N, n1=max(2, N // 10), n2=max(2, N // 100), n3=c["n3"] if i % 2 else 0,
                   mobility=float(rng.uniform(0.03, 0.1)))
        out.append(_panel(sub, int(rng.integers(1 << 31)), K=K))
    return out


def _keys(c, seed):
    """Raw int64 keys of a panel's workers and firms: ids with gaps, as files hold them."""
    p = _panel(dict(c, shape="worker_firm", K=1, weights=False), seed)
    return p["refs"][0] * 7 + 100_003, p["refs"][1] * 3 + 11


# ---------------------------------------------------------------------------
# the measured calls
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "group":
        return {"case": c, "keys": [_host(k) for k in _keys(c, seed)]}
    if kind == "panels":
        ps = _uneven(c, seed)
        solvers = [api.FixedEffectSolverROCm(_fes(p), _host(p["w"])) for p in ps]
        Y = torch.cat([p["Y"].reshape(-1) for p in ps])
        start = np.concatenate([[0], np.cumsum([p["Y"].numel() for p in ps])])
        return {"case": c, "solvers": solvers, "Y": Y, "work": torch.empty_like(Y), "start": start[:-1],
                "K": [p["Y"].shape[0] for p in ps], "N": [p["Y"].shape[1] for p in ps]}
    p = _panel(c, seed)
    fes = _fes(p)
    s = {"case": c, "fes": fes, "w": _host(p["w"])}
    if kind == "resident":
        s["solver"] = api.FixedEffectSolverROCm(fes, s["w"], c["precision"], algorithm=c["algorithm"])
        s["Y"], s["work"] = p["Y"], torch.empty_like(p["Y"])
        return s
    Y = _host(p["Y"])
    if c["precision"] == "fp32":
        Y = Y.astype(np.float32)
    s["Y"] = [Y[k] for k in range(c["K"])]
    s["cols"] = [np.empty(c["N"], np.float64) for _ in range(c["K"])]
    if kind in ("host", "reweight"):
        s["solver"] = api.FixedEffectSolverROCm(fes, None if kind == "reweight" else s["w"], c["precision"],
                                                algorithm=c["algorithm"])
    return s


def _fill(s):
    for col, y in zip(s["cols"], s["Y"]):
        np.copyto(col, y)
    return s["cols"]


def run(state):
    s, c = state, state["case"]
    kind, K = c["kind"], c["K"]
    tol = TOL32 if c["precision"] == "fp32" else TOL64
    if kind == "group":
        fe = api.FixedEffect(*s["keys"], device=True)
        return {"refs": fe.refs, "n": fe.n}
    if kind == "panels":
        s["work"].copy_(s["Y"])
        torch.cuda.current_stream().synchronize()  # the library's streams do not wait for torch's
        _, conv = api.solve_residuals_panels(s["solvers"], [s["work"].data_ptr() + 8 * int(o) for o in s["start"]],
                                             s["K"], s["N"], TOL64, MAXITER)
        return {"residuals": s["work"], "converged": np.concatenate(conv)}
    if kind == "resident":
        s["work"].copy_(s["Y"])
        torch.cuda.current_stream().synchronize()
        _, conv = s["solver"].solve_residuals_device(s["work"].data_ptr(), K, c["N"], tol, MAXITER)
        return {"residuals": s["work"], "converged": conv}
    if kind == "coefficients":
        obs, _, conv = api.solve_coefficients(s["Y"][0], s["fes"], s["w"], double_precision=True, tol=tol,
                                              maxiter=MAXITER)
        return {"coefficients": obs, "converged": conv}
    cols = _fill(s)
    if kind == "call":
        target = cols if K > 1 else cols[0]
        _, _, conv = api.solve_residuals(target, s["fes"], s["w"], double_precision=c["precision"] != "fp32", tol=tol,
                                         maxiter=MAXITER, progress_bar=False)
    else:
        if kind == "reweight":
            s["solver"].update_weights(s["w"])
        _, _, conv = s["solver"].solve_residuals_many(cols, tol, MAXITER)
    if c["precision"] == "fp32":  # the caller's vectors are Float32: they come back as such
        return {"residuals": [col.astype(np.float32) for col in cols], "converged": conv}
    return {"residuals": cols, "converged": conv}


def work(case):
    """Each input read once and each output written once: one pass of a solve cannot do without these."""
    c = case
    G = 3 if c["n3"] else 2
    if c["kind"] == "group":
        return {"bytes": 3 * 8 * c["N"], "flops": 0}
    if c["kind"] == "panels":
        one = [work(dict(c, kind="resident", N=N, K=K, n3=c["n3"] if i % 2 else 0))
               for i, (N, K) in enumerate(_sizes(c))]
        return {k: sum(o[k] for o in one) for k in ("bytes", "flops")}
    N, K = c["N"], c["K"]
    s = 4 if c["precision"] == "fp32" else 8
    per_obs = 4 * G + (8 if c["weights"] else 0) + (8 if c["interacted"] else 0)
    out = G * 8 if c["kind"] == "coefficients" else K * s
    return {"bytes": N * (per_obs + K * s + out), "flops": 2 * G * N * K}


# ---------------------------------------------------------------------------
# the same results in 64 bits, by plain torch
# ---------------------------------------------------------------------------
_FEW, _CHUNK = 128, 4096


def _rows(i, j, v, shape):
    """The sparse matrix with v[k] at (i[k], j[k]) (no pair twice), by rows."""
    order = torch.argsort(i)
    start = torch.zeros(shape[0] + 1, dtype=torch.int64, device=i.device)
    start[1:] = torch.cumsum(torch.bincount(i, minlength=shape[0]), 0)
    return torch.sparse_csr_tensor(start, j[order], v[order], shape)


def _least_squares(p, iterations=2000):
    """Level coefficients X[g] (n_g x K) and residuals (K x N) of the weighted least squares of Y on the fixed effects:
    conjugate gradients on the normal equations, whose cells are summed once per pair of levels."""
    refs, n, Y = p["refs"], p["n"], p["Y"].to(torch.float64).T.contiguous()
    N, G = Y.shape[0], len(refs)
    one = torch.ones(N, dtype=torch.float64, device=Y.device)
    w = one if p["w"] is None else p["w"]
    z = [one if zz is None else zz for zz in p["z"]]
    rows = torch.arange(N, device=Y.device)
    A = [_rows(refs[g], rows, w * z[g], (n[g], N)) for g in range(G)]  # the adjoint of each effect's map, weighted
    d = [1 / torch.sqrt(A[g] @ z[g][:, None]) for g in range(G)]
    blocks = {}
    for a in range(G):
        for b in range(a + 1, G):
            u, cell = torch.unique(refs[a] * n[b] + refs[b], return_inverse=True)
            v = (_rows(cell, rows, w * z[a] * z[b], (len(u), N)) @ one[:, None])[:, 0]
            i, j = u // n[b], u % n[b]
            v = v * d[a][i, 0] * d[b][j, 0]
            if n[b] <= _FEW:
                m = torch.zeros(-(-n[a] // _CHUNK) * _CHUNK, n[b], dtype=torch.float64, device=Y.device)
                m[i, j] = v
                blocks[a, b] = m[:n[a]], m.reshape(-1, _CHUNK, n[b]).transpose(1, 2).contiguous()
            else:
                blocks[a, b] = _rows(i, j, v, (n[a], n[b])), _rows(j, i, v, (n[b], n[a]))

    def normal(x):
        y = [t.clone() for t in x]
        for (a, b), (m, mt) in blocks.items():
            y[a] += m @ x[b]
            if mt.dim() == 3:  # a block of rows at a time: the product is much longer than wide
                xa = torch.zeros(mt.shape[0] * _CHUNK, x[a].shape[1], dtype=x[a].dtype, device=x[a].device)
                xa[:n[a]] = x[a]
                y[b] += torch.bmm(mt, xa.reshape(-1, _CHUNK, xa.shape[1])).sum(0)
            else:
                y[b] += mt @ x[a]
        return y

    def dot(x, y):
        return sum((s * t).sum(0) for s, t in zip(x, y))

    def ratio(a, b):
        return torch.where(b > 0, a / b, torch.zeros_like(a))

    r = [d[g] * (A[g] @ Y) for g in range(G)]
    del A
    x, s, rr = [torch.zeros_like(t) for t in r], [t.clone() for t in r], dot(r, r)
    stop = rr * 1e-13 ** 2
    for it in range(iterations):
        q = normal(s)
        alpha = ratio(rr, dot(s, q))
        for g in range(G):
            x[g] += alpha * s[g]
            r[g] -= alpha * q[g]
        new = dot(r, r)
        if it % 10 == 9 and bool((new <= stop).all()):
            break
        beta = ratio(new, rr)
        s, rr = [t + beta * u for t, u in zip(r, s)], new
    for g in range(G):
        x[g] *= d[g]
        Y -= z[g][:, None] * x[g][refs[g]]
    return x, Y.T.contiguous()


def exact(case, seed):
    c = case
    if c["kind"] == "group":
        return None
    if c["kind"] == "panels":
        return {"residuals": torch.cat([_least_squares(p)[1].reshape(-1) for p in _uneven(c, seed)]), "converged": None}
    p = _panel(c, seed)
    if c["precision"] == "fp32":
        p["Y"] = p["Y"].to(torch.float32).to(torch.float64)
    x, r = _least_squares(p)
    if c["kind"] == "coefficients":  # one component: the second effect's mean over its levels moves to the first
        m = x[1].mean()
        full = [(x[0] + m)[p["refs"][0], 0], (x[1] - m)[p["refs"][1], 0]]
        return {"coefficients": [_host(v) for v in full], "converged": None}
    if c["kind"] == "resident":
        return {"residuals": r, "converged": None}
    return {"residuals": [_host(v) for v in r], "converged": None}
