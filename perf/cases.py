"""Timed workloads of the multiplication & solve library, called through its public entry points.

Each kind of case is one call (or the few calls) that a program using the library makes:

  gemm        C = op(A) op(B)              bzg_dgemm_ex / bzg_sgemm_ex
  gemm_split  C = A B, FP64-accurate       bzg_dgemm_fp64acc_i8 (automatic slice count)
  gemv        y = A x, y = trans(A) x      bzg_dgemv / bzg_sgemv and their _t forms
  laplace     y = S x, short rows          bzg_dsellmv / bzg_ssellmv on a packed plan
  zipf        y = S x, power-law rows      bzg_dcsrmv / bzg_scsrmv on a plan
  cg          conjugate gradients          bzg_dcg on a packed plan
  solve       one system A X = B           bzg_dgesv
  batch       many systems, FP64           bzg_dgesv_batched
  mixed       many systems, FP32 + refine  bzg_dsgesv_batched

Plans and contexts are made in `prepare`, where a program keeps them.  The FP64 solvers overwrite
A and B, so a pass starts by copying both into the working arrays, as `solve(A, x, b)` does.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import blaze_amd as bz
from blaze_amd import solve as bsolve

DEV = "cuda"
_DTYPE = {"f64": torch.float64, "f32": torch.float32}
_ctx = None


def listed():
    return [
        # the plain product at the size of the reference's own small dense benchmark: latency-bound
        dict(name="gemm-fp64-512", kind="gemm", dtype="f64", ta=False, tb=False, m=512, n=512, k=512, pad=0),
        # single-precision product of a column-major operand, no size a multiple of a tile
        dict(name="gemm-fp32-ragged", kind="gemm", dtype="f32", ta=False, tb=True, m=1523, n=2021, k=1777, pad=3),
        # the largest product of the served mix
        dict(name="gemm-fp64-4096", kind="gemm", dtype="f64", ta=False, tb=False, m=4096, n=4096, k=4096, pad=0),
        # the FP64-accurate product from INT8 slices at the same size
        dict(name="gemm-split-4096", kind="gemm_split", m=4096, n=4096, k=4096, sigma=0.0),
        # a small matrix-vector product: one launch, little to read
        dict(name="gemv-fp64-small", kind="gemv", dtype="f64", trans=False, m=500, n=700),
        # a column-major (transposed) single-precision product from memory
        dict(name="gemv-t-fp32-large", kind="gemv", dtype="f32", trans=True, m=16384, n=12289),
        # 7-point Laplacian on a 128^3 grid: the stencil SpMV
        dict(name="spmv-laplace128", kind="laplace", dtype="f64", nx=128),
        # power-law row lengths (Zipf s = 1.5, 1..2000 per row), random columns: the graph SpMV
        dict(name="spmv-zipf-1e6", kind="zipf", dtype="f64", n=1000000),
        # conjugate gradients on the 5-point Laplacian, vectors of 8 MB
        dict(name="cg-1000", kind="cg", nx=1000, iterations=50),
        # one system too large for the batched solvers, several right-hand sides
        dict(name="solve-3000", kind="solve", n=3000, nrhs=16),
        # many small systems, orders 4..256 and 1..8 right-hand sides, half of them with interchanges
        dict(name="batch-fp64-10000", kind="batch", count=10000, nmax=256),
        # the same orders in mixed precision to 1e-12, 10 % of the systems with condition number 1e8
        dict(name="batch-mixed-10000", kind="mixed", count=10000, nmax=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm_split", "gemv", "laplace", "zipf", "cg", "solve", "batch", "mixed"])
    if kind == "gemm":
        return dict(kind=kind, dtype=rng.choice(["f64", "f32"]), ta=rng.random() < 0.25, tb=rng.random() < 0.25,
                    m=_log_int(rng, 32, 4096), n=_log_int(rng, 32, 4096), k=_log_int(rng, 32, 4096),
                    pad=rng.choice([0, 0, 1, 8]))
    if kind == "gemm_split":
        return dict(kind=kind, m=_log_int(rng, 1024, 4096), n=_log_int(rng, 1024, 4096), k=_log_int(rng, 1024, 4096),
                    sigma=rng.choice([0.0, 0.0, 4.0]))
    if kind == "gemv":
        return dict(kind=kind, dtype=rng.choice(["f64", "f32"]), trans=rng.random() < 0.5, m=_log_int(rng, 64, 16384),
                    n=_log_int(rng, 64, 12289))
    if kind == "laplace":
        return dict(kind=kind, dtype=rng.choice(["f64", "f32"]), nx=_log_int(rng, 24, 128))
    if kind == "zipf":
        return dict(kind=kind, dtype=rng.choice(["f64", "f32"]), n=_log_int(rng, 20000, 1000000))
    if kind == "cg":
        return dict(kind=kind, nx=_log_int(rng, 100, 1000), iterations=50)
    if kind == "solve":
        return dict(kind=kind, n=_log_int(rng, 200, 3000), nrhs=_log_int(rng, 1, 64))
    return dict(kind=kind, count=_log_int(rng, 300, 10000), nmax=_log_int(rng, 16, 256))


# ---- inputs -------------------------------------------------------------------------------------
def _context():
    global _ctx
    if _ctx is None:
        _ctx = bz.Context(stream=torch.cuda.current_stream().cuda_stream)
    return _ctx


def _p(t):
    return C.c_void_p(t.data_ptr())


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _uniform(g, shape, dtype=torch.float64):
    """Uniform on [-1, 1)."""
    return torch.rand(shape, generator=g, device=DEV, dtype=dtype).mul_(2).sub_(1)


def _gemm_inputs(case, seed):
    g = _gen(seed)
    dt = _DTYPE[case["dtype"]]
    m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
    A = _uniform(g, ((k, m) if case["ta"] else (m, k)), dt)
    B = _uniform(g, ((n, k) if case["tb"] else (k, n)), dt)
    # rows with `pad` elements of spacing, as a container with padded rows stores them
    Ap = torch.zeros((A.shape[0], A.shape[1] + pad), device=DEV, dtype=dt)
    Bp = torch.zeros((B.shape[0], B.shape[1] + pad), device=DEV, dtype=dt)
    Ap[:, :A.shape[1]] = A
    Bp[:, :B.shape[1]] = B
    return Ap, Bp


def _split_inputs(case, seed):
    """u 2^e with u uniform on [-1, 1) and e = round(N(0, sigma))."""
    g = _gen(seed)

    def one(shape):
        u = _uniform(g, shape)
        if case["sigma"] > 0:
            e = torch.randn(shape, generator=g, device=DEV, dtype=torch.float64).mul_(case["sigma"]).round_()
            u = torch.ldexp(u, e)
        return u

    return one((case["m"], case["k"])), one((case["k"], case["n"]))


def _gemv_inputs(case, seed):
    g = _gen(seed)
    dt = _DTYPE[case["dtype"]]
    A = _uniform(g, (case["m"], case["n"]), dt)
    x = _uniform(g, (case["m"] if case["trans"] else case["n"],), dt)
    return A, x


def _stencil(dims, diag, dtype):
    """CSR of the (2 d + 1)-point Laplacian on a d-dimensional grid, columns ascending."""
    n = math.prod(dims)
    idx = torch.arange(n, device=DEV, dtype=torch.int64)
    strides = [math.prod(dims[a + 1:]) for a in range(len(dims))]
    cols, keep, vals = [], [], []
    for sign in (-1, 1):
        for a in (range(len(dims)) if sign < 0 else reversed(range(len(dims)))):
            pos = (idx // strides[a]) % dims[a]
            keep.append(pos > 0 if sign < 0 else pos < dims[a] - 1)
            cols.append(idx + sign * strides[a])
            vals.append(torch.full((n,), -1.0, device=DEV, dtype=dtype))
        if sign < 0:
            keep.append(torch.ones(n, device=DEV, dtype=torch.bool))
            cols.append(idx)
            vals.append(torch.full((n,), diag, device=DEV, dtype=dtype))
    keep = torch.stack(keep, 1)
    rowptr = torch.zeros(n + 1, device=DEV, dtype=torch.int64)
    rowptr[1:] = torch.cumsum(keep.sum(1), 0)
    col = torch.stack(cols, 1)[keep].to(torch.int32)
    val = torch.stack(vals, 1)[keep].contiguous()
    return rowptr.to(torch.int32), col, val


def _laplace_inputs(case, seed):
    g = _gen(seed)
    dt = _DTYPE[case["dtype"]]
    nx = case["nx"]
    rp, ci, va = _stencil([nx, nx, nx], 6.0, dt)
    return rp, ci, va, _uniform(g, (nx ** 3,), dt)


def _zipf_inputs(case, seed):
    """Row lengths with P(len = l) ~ l^-1.5 on 1..2000; a row's columns are ascending, one from
    each of `len` equal parts of the column range; values N(0, 1), x uniform."""
    g = _gen(seed)
    dt = _DTYPE[case["dtype"]]
    n = case["n"]
    w = torch.arange(1, 2001, device=DEV, dtype=torch.float64).pow_(-1.5)
    cdf = torch.cumsum(w, 0) / w.sum()
    ln = torch.searchsorted(cdf, torch.rand(n, generator=g, device=DEV, dtype=torch.float64)).clamp_(max=1999) + 1
    rowptr = torch.zeros(n + 1, device=DEV, dtype=torch.int64)
    rowptr[1:] = torch.cumsum(ln, 0)
    nnz = int(rowptr[-1])
    row = torch.repeat_interleave(torch.arange(n, device=DEV), ln)
    k = torch.arange(nnz, device=DEV) - rowptr[row]
    length = ln[row]
    lo, hi = k * n // length, (k + 1) * n // length
    u = torch.rand(nnz, generator=g, device=DEV, dtype=torch.float64)
    col = lo + torch.minimum((u * (hi - lo)).to(torch.int64), hi - lo - 1)
    val = torch.randn(nnz, generator=g, device=DEV, dtype=dt)
    return rowptr.to(torch.int32), col.to(torch.int32), val, _uniform(g, (n,), dt)


def _cg_inputs(case, seed):
    g = _gen(seed)
    nx = case["nx"]
    rp, ci, va = _stencil([nx, nx], 4.0, torch.float64)
    return rp, ci, va, _uniform(g, (nx * nx,))


def _solve_inputs(case, seed):
    g = _gen(seed)
    return _uniform(g, (case["n"], case["n"])), _uniform(g, (case["n"], case["nrhs"]))


def _haar(g, n, nmax):
    """[len(n), nmax, nmax] orthogonal matrices, Haar-distributed in their leading n x n blocks
    (products of the reflections of Gaussian vectors with falling support), identity elsewhere."""
    b = n.numel()
    Q = torch.eye(nmax, device=DEV, dtype=torch.float64).repeat(b, 1, 1)
    V = torch.randn((b, nmax, nmax), generator=g, device=DEV, dtype=torch.float64)
    j = torch.arange(nmax, device=DEV)
    for s in range(nmax - 1):
        on = (j[None, :] >= s) & (j[None, :] < n[:, None])
        v = torch.where(on, V[:, s], 0.0)
        v = v / v.norm(dim=1, keepdim=True).clamp_min(1e-300)
        Q = torch.baddbmm(Q, v[:, :, None], torch.bmm(v[:, None, :], Q), alpha=-2.0)
    return Q


def _batch_inputs(case, seed):
    """Orders uniform in 4..nmax, 1..8 right-hand sides.  batch: R + n I (R uniform on [-1, 1)), and
    every second of them with its rows rotated by half, every tenth system plain R: these need their
    interchanges.  mixed: R + n I, and every tenth system Q1 diag(logspace(0, -8)) Q2 with
    Haar-distributed Q1, Q2."""
    g = _gen(seed)
    count, nmax = case["count"], case["nmax"]
    r = np.random.default_rng([count, nmax])  # the orders belong to the case, the values to the seed
    n = r.integers(4, nmax + 1, count).astype(np.int32)
    nrhs = r.integers(1, 9, count).astype(np.int32)
    n64 = n.astype(np.int64)
    a_off, b_off, p_off = (np.concatenate([[0], np.cumsum(s)]) for s in (n64 * n64, n64 * nrhs, n64))
    A = _uniform(g, (int(a_off[-1]),))
    B = _uniform(g, (int(b_off[-1]),))
    sys_of = torch.from_numpy(np.repeat(np.arange(count), n)).to(DEV)
    i = torch.arange(int(p_off[-1]), device=DEV) - torch.from_numpy(p_off[:-1]).to(DEV)[sys_of]
    dn = torch.from_numpy(n64).to(DEV)
    order = dn[sys_of]
    shift, big = order.to(torch.float64), i
    if case["kind"] == "batch":
        shift = torch.where(sys_of % 10 == 9, 0.0, shift)
        big = torch.where(sys_of % 2 == 1, (i + order // 2) % order, i)
    A[torch.from_numpy(a_off[:-1]).to(DEV)[sys_of] + i * order + big] += shift
    if case["kind"] == "mixed":
        for h0 in range(0, count, 4000):  # 400 hard systems at a time
            hard = np.arange(h0, min(count, h0 + 4000), 10)
            hn = dn[torch.from_numpy(hard).to(DEV)]
            top = int(n[hard].max())
            j = torch.arange(top, device=DEV, dtype=torch.float64)
            sv = torch.pow(10.0, -8.0 * j[None, :] / (hn[:, None] - 1))
            M = torch.bmm(_haar(g, hn, top) * sv[:, None, :], _haar(g, hn, top))
            inside = (j[None, :] < hn[:, None])
            at = torch.cat([torch.arange(int(a_off[s]), int(a_off[s + 1])) for s in hard]).to(DEV)
            A[at] = M[inside[:, :, None] & inside[:, None, :]]
    return n, nrhs, a_off[:-1].copy(), b_off[:-1].copy(), p_off[:-1].copy(), A, B


def _plan(ctx, rp, n):
    plan = C.c_void_p()
    h = rp.cpu().numpy()
    ctx.call("bzg_csr_plan_create", n, n, h.ctypes.data_as(C.c_void_p), C.byref(plan))
    return plan


class _Plan:
    """Owns a plan handle; freed with the state that holds it."""

    def __init__(self, handle):
        self.handle = handle

    def __del__(self):
        torch.cuda.synchronize()
        bz.lib().bzg_csr_plan_destroy(self.handle)


def prepare(case, seed):
    ctx = _context()
    kind = case["kind"]
    st = {"kind": kind, "ctx": ctx, "case": case}
    if kind == "gemm":
        st["A"], st["B"] = _gemm_inputs(case, seed)
        st["C"] = torch.empty((case["m"], case["n"]), device=DEV, dtype=_DTYPE[case["dtype"]])
    elif kind == "gemm_split":
        st["A"], st["B"] = _split_inputs(case, seed)
        st["C"] = torch.empty((case["m"], case["n"]), device=DEV, dtype=torch.float64)
    elif kind == "gemv":
        st["A"], st["x"] = _gemv_inputs(case, seed)
        st["y"] = torch.empty(case["n"] if case["trans"] else case["m"], device=DEV, dtype=st["A"].dtype)
    elif kind in ("laplace", "zipf", "cg"):
        make = {"laplace": _laplace_inputs, "zipf": _zipf_inputs, "cg": _cg_inputs}[kind]
        rp, ci, va, x = make(case, seed)
        st.update(rp=rp, ci=ci, va=va, x=x, y=torch.empty_like(x))
        st["plan"] = _Plan(_plan(ctx, rp, x.numel()))
        if kind != "zipf":
            ctx.call("bzg_csr_plan_pack_sell", st["plan"].handle, _p(rp), _p(ci), _p(va),
                     0 if va.dtype == torch.float64 else 1)
    elif kind == "solve":
        st["A"], st["B"] = _solve_inputs(case, seed)
        st["LU"], st["X"] = torch.empty_like(st["A"]), torch.empty_like(st["B"])
        st["ipiv"] = torch.zeros(case["n"], device=DEV, dtype=torch.int32)
        st["info"] = torch.zeros(1, device=DEV, dtype=torch.int32)
    else:
        n, nrhs, a_off, b_off, p_off, A, B = _batch_inputs(case, seed)
        st.update(A=A, B=B, X=torch.empty_like(B))
        st["dev"] = [torch.from_numpy(v).to(DEV) for v in (n, nrhs, a_off, b_off, p_off)]
        st["order"] = bsolve.order_longest_first(ctx, n)
        st["info"] = torch.zeros(case["count"], device=DEV, dtype=torch.int32)
        if kind == "batch":
            st["LU"] = torch.empty_like(A)
            st["ipiv"] = torch.zeros(int(n.sum()), device=DEV, dtype=torch.int32)
        else:
            st["iter"] = torch.zeros(case["count"], device=DEV, dtype=torch.int32)
    return st


def run(st):
    ctx, case, kind = st["ctx"], st["case"], st["kind"]
    if kind == "gemm":
        f = "bzg_dgemm_ex" if case["dtype"] == "f64" else "bzg_sgemm_ex"
        A, B, Cm = st["A"], st["B"], st["C"]
        ctx.call(f, int(case["ta"]), int(case["tb"]), case["m"], case["n"], case["k"], 1.0, _p(A), A.shape[1],
                 _p(B), B.shape[1], 0.0, _p(Cm), case["n"])
        return Cm
    if kind == "gemm_split":
        ctx.call("bzg_dgemm_fp64acc_i8", case["m"], case["n"], case["k"], _p(st["A"]), case["k"], _p(st["B"]),
                 case["n"], _p(st["C"]), case["n"], 0)
        return st["C"]
    if kind == "gemv":
        f = "bzg_" + ("d" if case["dtype"] == "f64" else "s") + ("gemv_t" if case["trans"] else "gemv")
        ctx.call(f, case["m"], case["n"], 1.0, _p(st["A"]), case["n"], _p(st["x"]), 0.0, _p(st["y"]))
        return st["y"]
    if kind == "laplace":
        f = "bzg_dsellmv" if case["dtype"] == "f64" else "bzg_ssellmv"
        ctx.call(f, st["plan"].handle, _p(st["x"]), _p(st["y"]))
        return st["y"]
    if kind == "zipf":
        f = "bzg_dcsrmv" if case["dtype"] == "f64" else "bzg_scsrmv"
        ctx.call(f, st["plan"].handle, _p(st["rp"]), _p(st["ci"]), _p(st["va"]), _p(st["x"]), _p(st["y"]))
        return st["y"]
    if kind == "cg":
        # b = the state's x; the iteration starts from zero
        st["y"].zero_()
        ctx.call("bzg_dcg", st["plan"].handle, st["x"].numel(), _p(st["rp"]), _p(st["ci"]), _p(st["va"]), _p(st["x"]),
                 _p(st["y"]), case["iterations"], C.c_void_p(0))
        return st["y"]
    if kind == "solve":
        n, nrhs = case["n"], case["nrhs"]
        st["LU"].copy_(st["A"])
        st["X"].copy_(st["B"])
        ctx.call("bzg_dgesv", n, nrhs, _p(st["LU"]), n, _p(st["ipiv"]), _p(st["X"]), nrhs, _p(st["info"]))
        return {"x": st["X"], "lu": st["LU"], "ipiv": st["ipiv"], "info": st["info"]}
    n, nrhs, a_off, b_off, p_off = (_p(t) for t in st["dev"])
    if kind == "batch":
        st["LU"].copy_(st["A"])
        st["X"].copy_(st["B"])
        ctx.call("bzg_dgesv_batched", case["count"], n, nrhs, a_off, b_off, p_off, _p(st["LU"]), _p(st["X"]),
                 _p(st["ipiv"]), _p(st["info"]), _p(st["order"]))
        return {"x": st["X"], "lu": st["LU"], "ipiv": st["ipiv"], "info": st["info"]}
    ctx.call("bzg_dsgesv_batched", case["count"], n, nrhs, a_off, b_off, _p(st["A"]), _p(st["B"]), _p(st["X"]),
             _p(st["iter"]), _p(st["info"]), 1e-12, 30, _p(st["order"]))
    return {"x": st["X"], "iter": st["iter"], "info": st["info"]}


# ---- the work a pass cannot do without ------------------------------------------------------------
def _zipf_mean():
    k = np.arange(1, 2001, dtype=np.float64)
    return float((k ** -0.5).sum() / (k ** -1.5).sum())


def work(case):
    kind = case["kind"]
    es = 8 if case.get("dtype", "f64") == "f64" else 4
    if kind in ("gemm", "gemm_split"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "gemv":
        m, n = case["m"], case["n"]
        return {"bytes": es * (m * n + m + n), "flops": 2 * m * n}
    if kind == "laplace":
        nx = case["nx"]
        n, nnz = nx ** 3, 7 * nx ** 3 - 6 * nx ** 2
        return {"bytes": nnz * (es + 4) + 2 * n * es, "flops": 2 * nnz}
    if kind == "zipf":
        n, nnz = case["n"], case["n"] * _zipf_mean()
        return {"bytes": nnz * (es + 4) + (n + 1) * 4 + 2 * n * es, "flops": 2 * nnz}
    if kind == "cg":
        nx, it = case["nx"], case["iterations"]
        n, nnz = nx * nx, 5 * nx * nx - 4 * nx
        # an iteration reads the matrix and reads and writes x, r and d; one product more at the start
        return {"bytes": it * (12 * nnz + 48 * n) + 12 * nnz + 24 * n, "flops": it * (2 * nnz + 10 * n) + 2 * nnz}
    if kind == "solve":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 8 * (2 * n * n + 2 * n * r), "flops": 2 / 3 * n ** 3 + 2 * n * n * r}
    # orders uniform in 4..nmax, 4.5 right-hand sides on average
    n = np.arange(4, case["nmax"] + 1, dtype=np.float64)
    passes = 2 if kind == "batch" else 1
    return {"bytes": case["count"] * float((8 * (passes * n * n + 2 * 4.5 * n)).mean()),
            "flops": case["count"] * float((2 / 3 * n ** 3 + 2 * 4.5 * n * n).mean())}


# ---- 64-bit values ----------------------------------------------------------------------------------
def _row_sums(rp, ci, va, x):
    """S x in double from the CSR arrays, on the host."""
    rp, ci, va, x = (t.cpu().numpy() for t in (rp, ci, va.double(), x.double()))
    p = np.concatenate([va * x[ci], [0.0]])
    return torch.from_numpy(np.where(rp[1:] > rp[:-1], np.add.reduceat(p, rp[:-1]), 0.0))


def _exact_cg(case, seed):
    """The same iteration on the grid itself."""
    _, _, _, b = _cg_inputs(case, seed)
    nx = case["nx"]

    def apply(v):
        g = v.view(nx, nx)
        out = 4.0 * g
        out[1:] -= g[:-1]
        out[:-1] -= g[1:]
        out[:, 1:] -= g[:, :-1]
        out[:, :-1] -= g[:, 1:]
        return out.reshape(-1)

    x = torch.zeros_like(b)
    r = apply(x) - b
    delta, d = torch.dot(r, r), -r
    for _ in range(case["iterations"]):
        h = apply(d)
        alpha = delta / torch.dot(d, h)
        x = x + alpha * d
        r = r + alpha * h
        beta = torch.dot(r, r)
        d = (beta / delta) * d - r
        delta = beta
    return x


def _exact_batch(case, seed):
    n, nrhs, a_off, b_off, _, A, B = _batch_inputs(case, seed)
    A, B = A.cpu().numpy(), B.cpu().numpy()
    X = np.empty_like(B)
    for i in range(case["count"]):
        m, r = int(n[i]), int(nrhs[i])
        a = A[a_off[i]:a_off[i] + m * m].reshape(m, m)
        b = B[b_off[i]:b_off[i] + m * r].reshape(m, r)
        X[b_off[i]:b_off[i] + m * r] = np.linalg.solve(a, b).reshape(-1)
    return X


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        A, B = _gemm_inputs(case, seed)
        pad = case["pad"]
        A, B = (t[:, :t.shape[1] - pad].cpu().double() for t in (A, B))
        return (A.t() if case["ta"] else A) @ (B.t() if case["tb"] else B)
    if kind == "gemm_split":
        A, B = _split_inputs(case, seed)
        return A.cpu() @ B.cpu()
    if kind == "gemv":
        A, x = _gemv_inputs(case, seed)
        A, x = A.cpu().double(), x.cpu().double()
        return (A.t() if case["trans"] else A) @ x
    if kind == "laplace":
        return _row_sums(*_laplace_inputs(case, seed))
    if kind == "zipf":
        return _row_sums(*_zipf_inputs(case, seed))
    if kind == "cg":
        return _exact_cg(case, seed)
    if kind == "solve":
        A, B = (t.cpu() for t in _solve_inputs(case, seed))
        LU, piv = torch.linalg.lu_factor(A)
        return {"x": torch.linalg.lu_solve(LU, piv, B), "lu": LU, "ipiv": None, "info": None}
    X = _exact_batch(case, seed)
    return {"x": X, "lu": None, "ipiv": None, "info": None} if kind == "batch" else {"x": X, "iter": None, "info": None}
