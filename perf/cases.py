"""Performance cases of the tiled SpMV, the solvers and the tile-precision policy.

A case is a dict of plain values; `prepare` builds what a program holds before
the call (the handle, vectors, the installed policy), `run` makes one pass
through the package's entry points, `exact` restates the result in 64 bits
with plain torch.  Matrices are the families that the package's generators,
tests and benchmark use:

  lap2d     2D 5-point Dirichlet Laplacian (nx * ny)
  lap3d     3D 7-point Laplacian with a log-uniform diagonal 6*10^(3U)
  convdiff  3D 7-point upwind convection-diffusion (nonsymmetric)
  knn       symmetrised 8-nearest-neighbour graph Laplacian + 1e-2 I
  powerlaw  Chung-Lu graph Laplacian (degree exponent 2.5, 15 entries a row)
            + `shift` I, hubs of up to tens of thousands of entries
"""
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mille-feuille_amd"))

import millefeuille as mf  # noqa: E402
from millefeuille import gen, policy  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # A small product on a graph with hub rows: one launch, all latency.
        dict(name="spmv_fp64_powerlaw_20k", op="spmv", matrix="powerlaw", n=20_011, shift=1.0),
        # The roofline product: 2.1M rows, 14.6M entries, every tile FP64.
        dict(name="spmv_fp64_lap3d_128", op="spmv", matrix="lap3d", nx=128, ny=128, nz=128),
        # A product at per-tile levels chosen from the quantisation errors, on
        # an irregular graph whose row count is no multiple of the tile edge.
        dict(name="spmv_levels_knn_150k", op="spmv_levels", matrix="knn", n=150_001),
        # The smallest solve: the 64 x 64 Laplacian, where launches and
        # grid-wide synchronisation count.
        dict(name="cg_fp64_lap2d_64", op="cg", matrix="lap2d", nx=64, ny=64, policy="fp64", tol=1e-10),
        # An ordinary FP64 solve on a box mesh with odd edges (893k rows).
        dict(name="cg_fp64_lap3d_odd", op="cg", matrix="lap3d", nx=117, ny=89, nz=86, policy="fp64", tol=1e-10),
        # The headline solve: learned per-tile precision, 2.1M rows.
        dict(name="cg_learned_lap3d_128", op="cg", matrix="lap3d", nx=128, ny=128, nz=128, policy="learned",
             tol=1e-10),
        # The rule policy (the default of the mixed reference-named entry
        # points) with its fallback, 262k rows.
        dict(name="cg_rule_lap3d_64", op="cg", matrix="lap3d", nx=64, ny=64, nz=64, policy="rule", tol=1e-10),
        # A graph with hub rows, whose heavy tile-rows are split over waves.
        dict(name="cg_fp64_powerlaw_200k", op="cg", matrix="powerlaw", n=200_003, shift=1.0, policy="fp64",
             tol=1e-10),
        # The nonsymmetric solver on the 1M-row convection-diffusion system.
        dict(name="bicgstab_learned_convdiff_100", op="bicgstab", matrix="convdiff", nx=100, ny=100, nz=100,
             policy="learned", tol=1e-12),
        # Many small systems, several right-hand sides each, one launch.
        dict(name="batch_errbound_knn_48x8", op="batch", matrix="knn", nsys=48, nlo=1000, nhi=16000, nrhs=8,
             policy="errbound", tol=1e-11),
        # One step of fitting the policy to a system: the features and labels
        # of its tiles, then loss and gradient of a sample batch.
        dict(name="policy_step_lap3d_80", op="policy", matrix="lap3d", nx=80, ny=80, nz=80, samples=100_000),
        # A matrix used once: host CSR to handle to the first product on the
        # host again, as a driver does for each file it reads.
        dict(name="setup_lap3d_90", op="setup", matrix="lap3d", nx=90, ny=91, nz=93),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """nx * ny * nz of about a log-uniform row count, with unequal edges."""
    e = math.exp(rng.uniform(math.log(lo), math.log(hi))) ** (1.0 / 3.0)
    a, b = rng.uniform(0.8, 1.0), rng.uniform(0.8, 1.0)
    return dict(nx=max(3, int(e * a)), ny=max(3, int(e * b)), nz=max(3, int(e)))


def draw(rng):
    op = rng.choice(["spmv", "spmv", "spmv_levels", "cg", "cg", "cg", "bicgstab", "batch", "policy", "setup"])
    if op in ("spmv", "spmv_levels"):
        m = rng.choice(["lap3d", "lap2d", "knn", "powerlaw"])
    elif op == "cg":
        m = rng.choice(["lap3d", "lap3d", "lap2d", "knn", "powerlaw"])
    elif op == "setup":
        m = rng.choice(["lap3d", "powerlaw"])
    else:
        m = {"bicgstab": "convdiff", "batch": "knn", "policy": "lap3d"}[op]
    c = dict(op=op, matrix=m)
    if op == "batch":
        nlo = _logu(rng, 500, 4000)
        c.update(nsys=rng.randint(3, 48), nlo=nlo, nhi=nlo * rng.randint(2, 4), nrhs=rng.randint(1, 8))
    elif m == "lap2d":
        e = _logu(rng, 64, 100 if op == "cg" else 1000)
        c.update(nx=e, ny=max(3, int(e * rng.uniform(0.7, 1.0))))
    elif m == "knn":
        c.update(n=_logu(rng, 4000, 150_000))
    elif m == "powerlaw":
        c.update(n=_logu(rng, 10_000, 200_000), shift=1.0)
    else:
        c.update(_box(rng, 8000, {"policy": 500_000, "setup": 760_000, "bicgstab": 1_000_000}.get(op, 2_000_000)))
    if op in ("cg", "bicgstab"):
        c.update(policy=rng.choice(["fp64", "errbound", "learned"]),
                 tol={"knn": 1e-11, "convdiff": 1e-12}.get(m, 1e-10))
    if op == "batch":
        c.update(policy=rng.choice(["fp64", "errbound"]), tol=1e-11)
    if op == "policy":
        c.update(samples=_logu(rng, 2000, 100_000))
    return c


# ---------------------------------------------------------------------------
# Matrices
# ---------------------------------------------------------------------------

def _stencil(shape, diag, neigh):
    """CSR of a box stencil, x fastest, columns ascending: diag (n values) and
    {axis: (value at -1, value at +1)}."""
    nx, ny, nz = shape
    n = nx * ny * nz
    i = torch.arange(n)
    pos = {0: i % nx, 1: (i // nx) % ny, 2: i // (nx * ny)}
    step = {0: 1, 1: nx, 2: nx * ny}
    axes = sorted(neigh)
    cols, keep, vals = [], [], []
    for d in reversed(axes):
        cols.append(i - step[d])
        keep.append(pos[d] > 0)
        vals.append(torch.full((n,), neigh[d][0], dtype=torch.float64))
    cols.append(i)
    keep.append(torch.ones(n, dtype=torch.bool))
    vals.append(diag)
    for d in axes:
        cols.append(i + step[d])
        keep.append(pos[d] < shape[d] - 1)
        vals.append(torch.full((n,), neigh[d][1], dtype=torch.float64))
    k = torch.stack(keep, 1)
    rp = torch.zeros(n + 1, dtype=torch.int64)
    rp[1:] = torch.cumsum(k.sum(1), 0)
    return (rp.to(torch.int32).numpy(), torch.stack(cols, 1)[k].to(torch.int32).numpy(),
            torch.stack(vals, 1)[k].numpy())


def _matrix(case, seed):
    m = case["matrix"]
    if m == "lap2d":
        n = case["nx"] * case["ny"]
        return _stencil((case["nx"], case["ny"], 1), torch.full((n,), 4.0, dtype=torch.float64),
                        {0: (-1.0, -1.0), 1: (-1.0, -1.0)})
    if m == "lap3d":
        n = case["nx"] * case["ny"] * case["nz"]
        g = torch.Generator().manual_seed(seed)
        diag = 6.0 * 10.0 ** (3.0 * torch.rand(n, generator=g, dtype=torch.float64))
        return _stencil((case["nx"], case["ny"], case["nz"]), diag, {d: (-1.0, -1.0) for d in range(3)})
    if m == "convdiff":
        # cell Peclet number 0.5, velocity (1, 0.5, 0.25), first-order upwind
        n = case["nx"] * case["ny"] * case["nz"]
        w = (1.0, 0.5, 0.25)
        return _stencil((case["nx"], case["ny"], case["nz"]),
                        torch.full((n,), 6.0 + sum(w), dtype=torch.float64),
                        {d: (-1.0 - w[d], -1.0) for d in range(3)})
    if m == "knn":
        return gen.knn_laplacian(case["n"], seed=seed)
    return gen.powerlaw_laplacian(case["n"], 15 * case["n"], seed=seed, shift=case["shift"])


def _rows(case):
    if "n" in case:
        return case["n"]
    return case["nx"] * case["ny"] * case.get("nz", 1)


def _systems(case, seed):
    """The batch's graphs: row counts evenly spread over the logarithm of [nlo, nhi]."""
    sizes = np.geomspace(case["nlo"], case["nhi"], case["nsys"])
    return [gen.knn_laplacian(int(n), seed=seed * 1000 + k) for k, n in enumerate(sizes)]


def _vector(n, seed, shape=None):
    """Values U[-1, 1] on the host."""
    g = torch.Generator().manual_seed(seed + 7919)
    return torch.rand(shape or (n,), generator=g, dtype=torch.float64) * 2.0 - 1.0


def _rhs(case, seed, csr):
    """Right-hand side: U[-1, 1]; for the convection-diffusion systems A x*
    with x* U[-1, 1]."""
    n = len(csr[0]) - 1
    v = _vector(n, seed)
    return _product(csr, v.to(DEV)).cpu() if case["matrix"] == "convdiff" else v


# ---------------------------------------------------------------------------
# State and passes
# ---------------------------------------------------------------------------

def _buf(t):
    """A torch tensor as the package takes a device array (its `ptr`)."""
    return SimpleNamespace(ptr=t.data_ptr(), tensor=t)


def _padded(tm, host, dtype=torch.float64):
    t = torch.zeros(tm.npad, dtype=dtype, device=DEV)
    if host is not None:
        t[: len(host)] = host.to(DEV, dtype)
    return t


def _levels(tm):
    """Cheapest payload within FP32 rounding of each tile's largest entry."""
    a = tm.arrays()
    big = np.maximum.reduceat(np.abs(a["Blockcsr_Val"]), a["csr_offset"][:-1])
    err = tm.quant_error()
    lv = np.full(tm.tilenum, 1, np.uint8)
    lv[err[1] <= 2.0 ** -24 * big] = 2
    lv[err[2] <= 2.0 ** -24 * big] = 3
    return lv


def prepare(case, seed):
    s = SimpleNamespace(case=case)
    op = case["op"]
    if op == "batch":
        s.systems = [mf.TiledMatrix(*a) for a in _systems(case, seed)]
        s.bs = [_vector(0, seed + 31 * k, (case["nrhs"], t.rowA)).numpy() for k, t in enumerate(s.systems)]
        return s
    csr = _matrix(case, seed)
    n = len(csr[0]) - 1
    if op == "setup":
        s.csr, s.x = csr, _vector(n, seed).numpy()
        return s
    s.tm = tm = mf.TiledMatrix(*csr)
    if op in ("spmv", "spmv_levels"):
        s.x = _buf(_padded(tm, _vector(n, seed)))
        s.y = _buf(_padded(tm, None))
        if op == "spmv_levels":
            tm.set_precision(_levels(tm))
            s.x32 = _buf(s.x.tensor.float())
    elif op == "policy":
        s.v = _buf(_padded(tm, _vector(n, seed)))
        s.params, s.feat, s.labels = _samples(case, seed)
    else:
        s.b = _buf(_padded(tm, _rhs(case, seed, csr)))
        s.x = _buf(_padded(tm, None))
        if case["policy"] == "learned":
            policy.install(tm, policy.load())
    return s


def _samples(case, seed):
    """Parameters, tile features and labels as a trace of systems gives them:
    few-entry to dense tiles, exact to coarse payloads, all stages of a solve."""
    n = case["samples"]
    rng = np.random.default_rng(seed)
    f = np.empty((n, 8), np.float32)
    f[:, 0] = rng.integers(1, 257, n) / 256.0
    f[:, 1] = rng.random(n) * 0.5
    f[:, 2] = -rng.random(n)
    f[:, 3] = -rng.random(n)
    f[:, 4] = rng.random(n)
    f[:, 5] = rng.uniform(-1, 1, n)
    f[:, 6] = rng.normal(0, 0.1, n)
    f[:, 7] = -rng.random(n) * 0.65
    lab = rng.integers(0, 4, n).astype(np.int32)
    return policy.init_params(seed), f, lab


def run(s):
    op = s.case["op"]
    if op == "spmv":
        s.tm.spmv(s.x, s.y)
        return s.y.tensor
    if op == "spmv_levels":
        s.tm.spmv(s.x, s.y, mode=1, d_x32=s.x32)
        return s.y.tensor
    if op in ("cg", "bicgstab"):
        s.x.tensor.zero_()
        getattr(s.tm, op)(s.b, s.x, tol=s.case["tol"], policy=s.case["policy"])
        return s.x.tensor
    if op == "batch":
        xs, _ = mf.batch_cg(s.systems, s.bs, nrhs=s.case["nrhs"], tol=s.case["tol"], policy=s.case["policy"])
        return xs
    if op == "policy":
        feat = policy.features(s.tm, s.v, 1e-3)
        lab = policy.labels(s.tm, s.v)
        loss, grad = policy.grad(s.params, s.feat, s.labels)
        return {"features": feat, "labels": lab, "logits": policy.forward(s.params, s.feat), "loss": loss, "grad": grad}
    tm = mf.TiledMatrix(*s.csr)
    x, y = tm.vector(s.x), tm.vector()
    tm.spmv(x, y)
    out = y.get(tm.rowA)
    for o in (x, y, tm):
        o.free()
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

_ROW_ENTRIES = {"lap2d": 5, "lap3d": 7, "convdiff": 7, "knn": 10.5, "powerlaw": 15}
_DIGIT_ITERS = {"lap2d": 13, "lap3d": 45, "convdiff": 21, "knn": 30, "powerlaw": 6}  # iterations per digit


def work(case):
    """One read of the matrix (value and a byte of column per entry) and of
    every vector an iteration needs, times the typical iterations to the
    tolerance."""
    op, per = case["op"], _ROW_ENTRIES[case["matrix"]]
    if op == "batch":
        n = case["nsys"] * (case["nhi"] - case["nlo"]) / math.log(case["nhi"] / case["nlo"])
        it = _DIGIT_ITERS["knn"] * -math.log10(case["tol"]) * case["nrhs"]
        return {"bytes": it * n * (per * 5 + 24), "flops": it * n * (2 * per + 10)}
    n = _rows(case)
    nnz = n * per
    if op == "spmv":
        return {"bytes": nnz * 9 + n * 16, "flops": 2 * nnz}
    if op == "spmv_levels":
        return {"bytes": nnz * 2.5 + n * 12, "flops": 2 * nnz}
    if op == "setup":
        return {"bytes": nnz * 12 + n * 20, "flops": 2 * nnz}
    if op == "policy":
        return {"bytes": nnz * 16 + n * 8 + nnz / 16 * 36 + case["samples"] * 52, "flops": case["samples"] * 8448 + 8 * nnz}
    it = (_DIGIT_ITERS[case["matrix"]] if case["matrix"] != "lap2d" else 0.21 * case["nx"]) * -math.log10(case["tol"])
    spmvs = 2 if op == "bicgstab" else 1
    size, vec = (9, 8) if case["policy"] == "fp64" else (5, 4)
    return {"bytes": it * spmvs * (nnz * size + n * 3 * vec), "flops": it * spmvs * (2 * nnz + 10 * n)}


# ---------------------------------------------------------------------------
# The results in 64 bits
# ---------------------------------------------------------------------------

def _product(csr, x):
    """A x with plain torch (x: a vector, or one column per right-hand side)."""
    rp, ci, va = (torch.from_numpy(np.asarray(a)).to(x.device) for a in csr)
    rows = torch.repeat_interleave(torch.arange(len(rp) - 1, device=x.device), rp.diff().long())
    v = va if x.dim() == 1 else va[:, None]
    return torch.zeros_like(x).index_add_(0, rows, v * x[ci.long()])


def _solve(csr, b):
    """The solution of an SPD system to rounding: conjugate gradients in 64
    bits, restarted from the recomputed residual until it no longer falls."""
    rp, ci, va = (torch.from_numpy(np.asarray(a)).to(b.device) for a in csr)
    n = len(rp) - 1
    a = torch.sparse_csr_tensor(rp.long(), ci.long(), va, (n, n))
    one = b.dim() == 1
    b = b[:, None] if one else b
    x = torch.zeros_like(b)
    bn = torch.linalg.vector_norm(b, dim=0)
    last = math.inf
    for _ in range(4):
        r = b - a @ x
        rel = float((torch.linalg.vector_norm(r, dim=0) / bn).max())
        if not rel < 0.1 * last or rel < 1e-15:
            break
        last = rel
        p = r.clone()
        rr = (r * r).sum(0)
        stop = rr * 1e-16
        for it in range(5000):
            q = a @ p
            al = rr / (p * q).sum(0)
            x += al * p
            r -= al * q
            new = (r * r).sum(0)
            if it % 16 == 15 and bool((new <= stop).all()):
                break
            p = r + (new / rr) * p
            rr = new
    return x[:, 0] if one else x


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        out = []
        for k, csr in enumerate(_systems(case, seed)):
            b = _vector(0, seed + 31 * k, (case["nrhs"], len(csr[0]) - 1))
            out.append(_solve(csr, b.T.contiguous().to(DEV)).T.contiguous())
        return out
    if op == "policy":
        loss, grad, z = _grad64(*_samples(case, seed))
        return {"features": None, "labels": None, "logits": z, "loss": loss, "grad": grad}
    csr = _matrix(case, seed)
    n = len(csr[0]) - 1
    v = _vector(n, seed).to(DEV)
    if op == "setup":
        return _product(csr, v)
    if op in ("spmv", "spmv_levels"):
        y = _product(csr, v)
    else:
        # (the convection-diffusion right-hand side is A v)
        y = v if op == "bicgstab" else _solve(csr, v)
    out = torch.zeros((n + 15) // 16 * 16, dtype=torch.float64, device=DEV)
    out[:n] = y
    return out


def _grad64(params, feat, labels):
    """Loss, gradient and logits of the 8-32-32-4 network, FP16 weights."""
    p = torch.from_numpy(params).half().double().to(DEV).requires_grad_(True)
    o, w = 0, []
    for i, k in ((8, 32), (32, 32), (32, 4)):
        w.append((p[o:o + i * k].view(k, i), p[o + i * k:o + i * k + k]))
        o += i * k + k
    h = torch.from_numpy(feat).double().to(DEV)
    for j, (a, c) in enumerate(w):
        h = h @ a.T + c
        h = torch.relu(h) if j < 2 else h
    loss = torch.nn.functional.cross_entropy(h, torch.from_numpy(labels).long().to(DEV))
    loss.backward()
    return float(loss), p.grad, h.detach()
