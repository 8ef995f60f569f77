"""Workloads of the eigensolver on one GPU, through its public entry points.

A case is a dict of plain values.  Its "kind" names the call:

  spmv     y = A x with the context's operator (Context.spmv)
  spmm     Y = A X for a block of vectors (Context.spmm)
  gram     C = V^T W of two tall panels (Context.gram)
  update   Y = V Q, the basis update of a restart (Context.tall_gemm)
  adjoint  eigenvalue gradients, the backward of autograd.eigvals (stored
           entries) and autograd.eigvals_potential (a diagonal potential)
  apply    one application of a multilevel ILDL preconditioner
           (Context.precond_apply)
  solve    a whole Jacobi-Davidson solve with the matrix and the
           preconditioner kept (Context.pjd), or in reverse communication
           with the diagonal preconditioner (Context.pjdrevcom)

and its "matrix" one of jadamilu_amd.matrices: "chain" (the tridiagonal
tridiag(5, i, 5) of the user guide's EXAMPLE9), "laplace" (Dirichlet, a 2D
or 3D box) or "anderson" (periodic cube, random potential, W = 16.5).
"""
import ctypes
import functools

import numpy as np
import torch

from jadamilu_amd import lib
from jadamilu_amd import matrices as M
from jadamilu_amd.ildl import IldlFactor
from jadamilu_amd.jd import Context, lx_optimal

F64 = torch.float64


def listed():
    return [
        # the smallest product: a thousand rows, bound by the launch
        dict(name="spmv_chain_1000", kind="spmv", matrix="chain", n=1000),
        # the product of the benchmark's matrix
        dict(name="spmv_laplace_128", kind="spmv", matrix="laplace", a=128, b=128, c=128),
        # a block of the ten wanted vectors on the largest Anderson matrix
        # (residual checks, block starts)
        dict(name="spmm_anderson_100_x10", kind="spmm", matrix="anderson", L=100, k=10),
        # the Rayleigh-Ritz block of a MADSPACE = 20 run at the benchmark's size
        dict(name="gram_128_20x20", kind="gram", n=128 ** 3, k=20, m=20),
        # an odd order with panels that fill no tile (a cluster against the
        # basis of a MADSPACE = 25 run)
        dict(name="gram_97_13x25", kind="gram", n=97 ** 3, k=13, m=25),
        # the restart of a MADSPACE = 20 run: 20 columns to 10
        dict(name="update_128_20to10", kind="update", n=128 ** 3, k=20, m=10),
        # the gradient of ten eigenvalues in the stored entries of the largest
        # Anderson matrix
        dict(name="adjoint_anderson_100_x10", kind="adjoint", L=100, k=10, potential=False),
        # one apply of a definite factor (FP64, the tuned sweep count)
        dict(name="apply_laplace_64", kind="apply", matrix="laplace", a=64, b=64, c=64,
             sweeps=4, single=False),
        # one apply of an indefinite factor stored in FP32 (the mixed path)
        dict(name="apply_anderson_32_fp32", kind="apply", matrix="anderson", L=32, sweeps=9,
             single=True),
        # the guide's diagonally preconditioned run: a thousand rows, every
        # inner step bound by launches and round trips
        dict(name="solve_chain_1000", kind="solve", matrix="chain", n=1000, neig=5),
        # a small 2D solve with the kept factor
        dict(name="solve_laplace_110x87", kind="solve", matrix="laplace", a=110, b=87, c=1,
             neig=5),
        # a whole solve with the kept factor: the benchmark's problem at a size
        # whose factor takes seconds
        dict(name="solve_laplace_73x61x51", kind="solve", matrix="laplace", a=73, b=61, c=51,
             neig=5),
    ]


def _log(rng, lo, hi):
    """A whole number spread over lo..hi in its logarithm."""
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def _drawn_matrix(rng, n_max):
    kind = rng.choice(["chain", "laplace", "laplace", "anderson", "anderson"])
    if kind == "chain":
        return dict(matrix="chain", n=_log(rng, 1000, min(n_max, 1000000)))
    if kind == "anderson":
        return dict(matrix="anderson", L=_log(rng, 10, int(n_max ** (1 / 3))))
    if rng.random() < 0.3:
        m = int(n_max ** 0.5)
        return dict(matrix="laplace", a=_log(rng, 32, m), b=_log(rng, 32, m), c=1)
    m = int(n_max ** (1 / 3))
    return dict(matrix="laplace", a=_log(rng, 10, m), b=_log(rng, 10, m), c=_log(rng, 10, m))


def draw(rng):
    kind = rng.choice(["spmv", "spmm", "gram", "update", "adjoint", "apply", "apply", "solve"])
    if kind == "spmv":
        return dict(kind=kind, **_drawn_matrix(rng, 128 ** 3))
    if kind == "spmm":
        return dict(kind=kind, **_drawn_matrix(rng, 100 ** 3), k=rng.randint(2, 10))
    if kind in ("gram", "update"):
        k, m = rng.randint(1, 32), rng.randint(1, 32)
        return dict(kind=kind, n=_log(rng, 1000, 128 ** 3 * 30 // (k + m) if k + m > 30
                                      else 128 ** 3), k=k, m=m)
    if kind == "adjoint":
        return dict(kind=kind, L=_log(rng, 10, 100), k=rng.randint(1, 10),
                    potential=rng.random() < 0.3)
    if kind == "apply":
        if rng.random() < 0.5:
            return dict(kind=kind, matrix="laplace", a=_log(rng, 16, 64), b=_log(rng, 16, 64),
                        c=_log(rng, 16, 64), sweeps=rng.randint(2, 6),
                        single=rng.random() < 0.5)
        return dict(kind=kind, matrix="anderson", L=_log(rng, 10, 32),
                    sweeps=rng.randint(6, 12), single=rng.random() < 0.5)
    if rng.random() < 0.3:
        return dict(kind=kind, matrix="chain", n=_log(rng, 500, 5000), neig=rng.randint(1, 5))
    # side ratios for which the lowest eigenvalues lie apart, so that the
    # vectors are determined to well below the tolerance
    if rng.random() < 0.5:
        a = _log(rng, 40, 160)
        return dict(kind=kind, matrix="laplace", a=a, b=round(0.79 * a), c=1,
                    neig=rng.randint(1, 5))
    a = _log(rng, 16, 70)
    return dict(kind=kind, matrix="laplace", a=a, b=round(0.84 * a), c=round(0.7 * a),
                neig=rng.randint(1, 5))


# ---- matrices and inputs ----------------------------------------------------

def _shape(case):
    return tuple(s for s in (case["a"], case["b"], case["c"]) if s > 1)


@functools.lru_cache(maxsize=4)
def _laplace(shape):
    return M.laplace(shape)


@functools.lru_cache(maxsize=2)
def _anderson(L):
    return M.anderson(L, 0.0, 0)  # the pattern and the hopping


def _matrix(case, seed):
    """1-based upper CSR (ia, ja, a), the diagonal first in every row."""
    if case["matrix"] == "laplace":
        return _laplace(_shape(case))
    if case["matrix"] == "chain":
        return M.tridiag(case["n"], np.arange(1, case["n"] + 1, dtype=float), 5.0)
    ia, ja, a = _anderson(case["L"])
    a = a.copy()
    a[ia[:-1] - 1] = M.anderson_potential(case["L"], 16.5, seed)
    return ia, ja, a


def _order(case):
    if "L" in case:
        return case["L"] ** 3
    return case["n"] if "n" in case else case["a"] * case["b"] * case["c"]


def _entries(case):
    """Stored entries of the upper triangle."""
    n = _order(case)
    if "L" in case:
        return 4 * n
    if case["matrix"] == "chain":
        return 2 * n - 1
    return n + sum(n - n // s for s in _shape(case))


def _normal(seed, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(*shape, dtype=F64, device="cuda", generator=g)


def _panels(case, seed):
    """Basis columns V (k x n, a row per column) and, for a Gram product, the
    images W (m x n) that go with them: each one of V's columns and a part
    outside of their span."""
    n, k, m = case["n"], case["k"], case["m"]
    V = _normal(seed, k, n) / n ** 0.5
    if case["kind"] == "update":
        Q = torch.linalg.qr(_normal(seed + 1, max(k, m), max(k, m)))[0][:m, :k].contiguous()
        return V, Q
    W = _normal(seed + 1, m, n) / n ** 0.5
    for j in range(m):
        W[j] += (1.0 + 0.1 * j) * V[j % k]
    return V, W


def _weights(case, seed):
    return np.random.default_rng(seed).standard_normal(case["k"])


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=dict(case))
    n = _order(case)
    if kind in ("gram", "update"):
        st["V"], st["W"] = _panels(case, seed)
        rows = (case["m"], case["k"]) if kind == "gram" else (case["m"], n)
        st["out"] = torch.empty(*rows, dtype=F64, device="cuda")
        st["ctx"] = Context(0)
    elif kind == "adjoint":
        st["X"] = _normal(seed, case["k"], n) / n ** 0.5
        st["w"] = _weights(case, seed)
        if not case["potential"]:
            ia, ja, _ = _anderson(case["L"])
            st["ia"] = torch.tensor(ia, dtype=torch.int32, device="cuda")
            st["ja"] = torch.tensor(ja, dtype=torch.int32, device="cuda")
        st["out"] = torch.empty(n if case["potential"] else ja.size, dtype=F64, device="cuda")
    elif kind in ("spmv", "spmm"):
        st["ctx"] = Context(0)
        st["ctx"].set_matrix(*_matrix(case, seed))
        k = case.get("k", 1)
        st["X"] = _normal(seed, k, n)
        st["out"] = torch.empty(k, n, dtype=F64, device="cuda")
    elif kind == "apply":
        st["ctx"] = Context(0)
        st["ctx"].attach_ildl(_factor(case, seed), sweeps=case["sweeps"])
        st["X"] = _normal(seed, n)
        st["out"] = torch.empty(n, dtype=F64, device="cuda")
    else:
        ctx = st["ctx"] = Context(0)
        st["stream"] = torch.cuda.ExternalStream(ctx.stream_ptr())
        ia, ja, a = _matrix(case, seed)
        st["x0"] = torch.tensor(np.random.default_rng(seed).random(n), device="cuda")
        st["X"] = torch.zeros(lx_optimal(n, case["neig"], 20), dtype=F64, device="cuda")
        torch.cuda.synchronize()
        if case["matrix"] == "chain":
            ctx.set_matrix(ia, ja, a)
            st["matrix"] = (a[ia[:-1] - 1], [-1], [-1])
        else:
            st["matrix"] = (a, ja, ia)
            _solve(st, 1)  # factors, tunes and keeps the preconditioner
    torch.cuda.synchronize()
    return st


def _factor(case, seed):
    ia, ja, a = _matrix(case, seed)
    return IldlFactor(ia.size - 1, ia, ja, a, droptol=1e-3, spd=case["matrix"] == "laplace",
                      single=case["single"])


def _solve(st, keep):
    """keep: ICNTL(2), 1 = set the preconditioner up, -1 = use the kept one."""
    case, ctx, X = st["case"], st["ctx"], st["X"]
    n = _order(case)
    with torch.cuda.stream(st["stream"]):
        X[:n].copy_(st["x0"])
    a, ja, ia = st["matrix"]
    if case["matrix"] == "chain":
        r = ctx.pjdrevcom(n, a, ja, ia, X.data_ptr(), X.numel(), neig=case["neig"], ninit=1,
                          madspace=20, maxiter=5000, tol=1e-10)
    else:
        r = ctx.pjd(n, a, ja, ia, X.data_ptr(), X.numel(), neig=case["neig"], isearch=1,
                    ninit=1, madspace=20, maxiter=5000, tol=1e-10, droptol=1e-3, mem=6.0,
                    icntl=(0, keep, 0, 0, 0))
    if r.info != 0:
        raise RuntimeError(f"solve: info {r.info}")
    return r.eigs, X[: n * r.neig].view(r.neig, n)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "solve":
        return _solve(st, -1)
    out = st["out"]
    if kind == "spmv":
        st["ctx"].spmv(st["X"].data_ptr(), out.data_ptr())
    elif kind == "spmm":
        n = st["X"].shape[1]
        st["ctx"].spmm(case["k"], st["X"].data_ptr(), n, out.data_ptr(), n)
    elif kind == "gram":
        n = case["n"]
        st["ctx"].gram(n, case["k"], case["m"], st["V"].data_ptr(), n, st["W"].data_ptr(), n,
                       out.data_ptr(), case["k"])
    elif kind == "update":
        n = case["n"]
        st["ctx"].tall_gemm(n, case["k"], case["m"], st["V"].data_ptr(), n, st["W"].data_ptr(),
                            case["k"], out.data_ptr(), n)
    elif kind == "apply":
        st["ctx"].precond_apply(out.data_ptr(), st["X"].data_ptr())
    else:
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        w = st["w"].ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        n, k = st["X"].shape[1], case["k"]
        if case["potential"]:
            rc = lib().jdhip_adjoint_diag(stream, n, st["X"].data_ptr(), n, k, w,
                                          out.data_ptr())
        else:
            rc = lib().jdhip_adjoint_csr(stream, n, st["ia"].data_ptr(), st["ja"].data_ptr(),
                                         st["X"].data_ptr(), n, k, w, out.data_ptr())
        if rc != 0:
            raise RuntimeError(f"adjoint: {rc}")
    return out


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    kind = case["kind"]
    n = _order(case)
    if kind == "gram":
        k, m = case["k"], case["m"]
        return dict(bytes=8 * (n * (k + m) + k * m), flops=2 * n * k * m)
    if kind == "update":
        k, m = case["k"], case["m"]
        return dict(bytes=8 * (n * (k + m) + k * m), flops=2 * n * k * m)
    if kind == "adjoint":
        k = case["k"]
        if case["potential"]:
            return dict(bytes=8 * n * (k + 1), flops=3 * n * k)
        return dict(bytes=12 * 4 * n + 4 * n + 8 * n * k, flops=3 * 4 * n * k)
    nnz = _entries(case)
    product = 12 * nnz + 4 * (n + 1)
    if kind in ("spmv", "spmm"):
        k = case.get("k", 1)
        return dict(bytes=product + 16 * n * k, flops=2 * (2 * nnz - n) * k)
    # the factor's entries over the matrix's, as its DROPTOL of 1e-3 gives them
    fill = 9.9 if case["matrix"] == "anderson" else 3.7
    value = 4 if case.get("single") else 8
    factor = int(fill * nnz) * (value + 4)
    if kind == "apply":
        # the factor read once, however many sweeps reuse it
        return dict(bytes=factor + 16 * n, flops=8 * case["sweeps"] * int(fill * nnz))
    # a solve: of the order of forty products and applies for each eigenpair
    steps = 40 * case["neig"]
    if case["matrix"] == "chain":
        return dict(bytes=steps * (product + 16 * n), flops=steps * 4 * nnz)
    return dict(bytes=steps * (product + factor + 32 * n),
                flops=steps * (4 + 32 * fill) * nnz)


def tolerance(case):
    """About four times what other kernel forms and 64-bit references of the
    same sums differ by, measured."""
    kind = case["kind"]
    if kind == "solve":
        # kernel forms change the vectors by 2e-13 at most, but what a solve
        # promises is a residual of 1e-10 over the gap to the next eigenvalue
        # (1e-4 and more on the boxes, of the order of 1 on the chain), which
        # is where another stopping step of the inner iteration ends
        return dict(rel=1e-9, max=1e-8) if case["matrix"] == "chain" else dict(rel=1e-6,
                                                                                max=1e-5)
    if kind == "gram":
        return dict(rel=1e-13, max=1e-12)  # sums of millions of terms, 3e-14
    if kind == "apply" and case["matrix"] == "anderson":
        return dict(rel=1e-14, max=4e-13)  # indefinite: sums that cancel, 2.4e-15
    if kind == "apply" and case["single"]:
        return dict(rel=2.5e-7, max=2e-6)  # FP32 work vectors, 6e-8
    return dict(rel=1e-15, max=4e-14)  # FP64 sums of a few terms, 2e-16


# ---- the same in plain 64-bit torch and numpy -------------------------------

def _times_upper(ia, ja, a, X):
    """(U + U^T - D) X for the stored upper triangle, X with a row a vector."""
    rows = torch.from_numpy(np.repeat(np.arange(ia.size - 1), np.diff(ia)))
    cols = torch.from_numpy(ja.astype(np.int64) - 1)
    v = torch.from_numpy(a)
    off = rows != cols
    Y = torch.zeros_like(X)
    for x, y in zip(X, Y):
        y.index_add_(0, rows, v * x[cols])
        y.index_add_(0, cols[off], v[off] * x[rows[off]])
    return Y


def _csr_times(ptr, idx, val, x):
    y = np.zeros(ptr.size - 1)
    np.add.at(y, np.repeat(np.arange(ptr.size - 1), np.diff(ptr)), val * x[idx])
    return y


def _csr_times_t(ptr, idx, val, x, n):
    y = np.zeros(n)
    np.add.at(y, idx, val * np.repeat(x, np.diff(ptr)))
    return y


def _solve_block(L, b, sweeps):
    """x = B^-1 b: `sweeps` Jacobi sweeps with L_B, D^-1, and with L_B^T."""
    lb = (L["lb_ptr"], L["lb_idx"], L["lb_val"])
    x = b
    for _ in range(sweeps):
        x = b - _csr_times(*lb, x)
    pair, d, o = L["dpair"], L["d"], L["doff"]
    p = np.where(pair >= 0, pair, 0)
    det = np.where(pair >= 0, d * d[p] - o * o, 1.0)
    b = np.where(pair >= 0, (d[p] * x - o * x[p]) / det, x / d)
    x = b
    for _ in range(sweeps):
        x = b - _csr_times_t(*lb, x, b.size)
    return x


def _apply_level(f, lev, r, sweeps):
    if lev == len(f["levels"]):
        return f["minv"] @ r
    L = f["levels"][lev]
    nB, perm = L["nB"], L["perm"]
    b = L["scal"][perm] * r[perm]
    lc = (L["lc_ptr"], L["lc_idx"], L["lc_val"])
    y = _solve_block(L, b[:nB], sweeps)
    z = b[nB:]
    if z.size:
        z = _apply_level(f, lev + 1, z - _csr_times(*lc, y), sweeps)
        y = y - _solve_block(L, _csr_times_t(*lc, z, nB), sweeps)
    out = np.empty(perm.size)
    out[perm] = L["scal"][perm] * np.concatenate([y, z])
    return out


def _box_eigs(shape, k):
    lam = np.zeros(1)
    for s in shape:
        one = 2.0 - 2.0 * np.cos(np.arange(1, s + 1) * np.pi / (s + 1))
        lam = np.sort((lam[:, None] + one[: k + 1]).ravel())[: k + 1]
    return lam[:k]


def exact(case, seed):
    kind = case["kind"]
    if kind == "gram":
        V, W = (t.cpu() for t in _panels(case, seed))
        return W @ V.T
    if kind == "update":
        V, Q = (t.cpu() for t in _panels(case, seed))
        return Q @ V
    if kind == "adjoint":
        X = (_normal(seed, case["k"], _order(case)) / _order(case) ** 0.5).cpu()
        w = torch.from_numpy(_weights(case, seed))
        if case["potential"]:
            return (w[:, None] * X * X).sum(0)
        ia, ja, _ = _anderson(case["L"])
        rows = torch.from_numpy(np.repeat(np.arange(ia.size - 1), np.diff(ia)))
        cols = torch.from_numpy(ja.astype(np.int64) - 1)
        g = sum(w[c] * X[c, rows] * X[c, cols] for c in range(case["k"]))
        return torch.where(rows == cols, g, 2.0 * g)
    if kind in ("spmv", "spmm"):
        X = _normal(seed, case.get("k", 1), _order(case)).cpu()
        return _times_upper(*_matrix(case, seed), X)
    if kind == "apply":
        f = _factor(case, seed).export()
        r = _normal(seed, _order(case)).cpu().numpy()
        return _apply_level(f, 0, r, case["sweeps"])
    if case["matrix"] == "laplace":
        return _box_eigs(_shape(case), case["neig"]), None
    n = case["n"]
    T = torch.diag(torch.arange(1, n + 1, dtype=F64))
    T += 5.0 * (torch.diag(torch.ones(n - 1, dtype=F64), 1)
                + torch.diag(torch.ones(n - 1, dtype=F64), -1))
    return torch.linalg.eigvalsh(T)[: case["neig"]].numpy(), None
