"""The diagonal form of the symmetric products against the CSR form of the same
matrix, and the matrices that must not take it.

Both forms add a row's m products in double in another order: each is off by
m * 2^-53 of the sum of absolute terms at most, so they agree to twice that (one
more for the rounding of that sum itself).
"""
import numpy as np
import pytest

from jadamilu_amd import matrices as M

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _products(mat, X, lanes):
    from jadamilu_amd.jd import Context
    ctx = Context(0)
    ctx.set_matrix(*mat, lanes_per_row=lanes)
    k, n = X.shape
    Y = torch.full((k + 1, n), 7.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ctx.spmv(X.data_ptr(), Y[0].data_ptr())
    ctx.spmm(k, X.data_ptr(), n, Y[1].data_ptr(), n)
    torch.cuda.synchronize()
    form = ctx.stats()["spmv_lanes"]
    ctx.close()
    return Y.cpu().numpy(), form


def _holes(n, seed):
    """Five diagonals with a fifth of the entries missing, rows in any order."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for d in (1, 7, 64, 1000):
        i = np.flatnonzero(rng.random(n - d) < 0.8)
        rows.append(i)
        cols.append(i + d)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    ia, ja, a = M.from_pairs(n, rows, cols, rng.standard_normal(rows.size),
                             rng.standard_normal(n))
    for i in range(0, n, 3):  # the diagonal anywhere in its row
        s = slice(ia[i] - 1, ia[i + 1] - 1)
        p = rng.permutation(s.stop - s.start)
        ja[s], a[s] = ja[s][p], a[s][p]
    return ia, ja, a


def _twice(n):
    """A path with one off-diagonal entry stored twice."""
    ia, ja, a = M.tridiag(n, 4.0, -1.0)
    at = ia[100] - 1 + 1
    ja, a = np.insert(ja, at, ja[at]), np.insert(a, at, 0.5)
    ia = ia.copy()
    ia[101:] += 1
    return ia, ja, a


def _many(n, m):
    """m diagonals above the main one."""
    d = 1 + 3 * np.arange(m)
    rows = np.concatenate([np.arange(n - k) for k in d])
    cols = np.concatenate([np.arange(n - k) + k for k in d])
    return M.from_pairs(n, rows, cols, np.cos(0.1 * np.arange(rows.size)), 2.0)


def _sparse_diagonals(n):
    """Diagonals that hold an entry in every 64th row only."""
    r = np.arange(0, n - 4000, 64)
    rows = np.concatenate([r] * 6)
    cols = np.concatenate([r + d for d in (1, 60, 900, 1500, 2100, 3900)])
    return M.from_pairs(n, rows, cols, np.ones(rows.size), 3.0)


@pytest.mark.parametrize("gen,diagonal", [
    (lambda: M.laplace((4096,)), True),
    (lambda: M.laplace((67, 63)), True),
    (lambda: M.laplace((67, 63), periodic=True), True),
    (lambda: M.laplace((17, 18, 19)), True),
    (lambda: M.anderson(17, 16.5, 3), True),
    (lambda: M.anderson(40, 16.5, 3), True),
    (lambda: M.from_pairs(5000, np.zeros(0, int), np.zeros(0, int), np.zeros(0),
                          np.arange(5000.0)), True),
    (lambda: _holes(4099, 1), True),
    (lambda: _many(5000, 6), True),
    (lambda: _many(5000, 7), False),
    (lambda: _many(5000, 15), False),
    (lambda: _many(5000, 16), False),
    (lambda: _sparse_diagonals(20000), False),
    (lambda: _twice(5000), False),
    (lambda: M.laplace((4095,)), False),
])
@pytest.mark.parametrize("k", [1, 2, 9, 10, 11, 21])
def test_diagonal_form_equals_csr(gen, diagonal, k):
    _dev()
    mat = gen()
    n = mat[0].size - 1
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    X = torch.randn(k, n, dtype=torch.float64, device="cuda:0", generator=g)
    y, form = _products(mat, X, 0)
    z, _ = _products(mat, X, 8)
    assert (form == -2) == diagonal
    scale, _ = _products((mat[0], mat[1], np.abs(mat[2])), X.abs(), 8)
    rows, cols = np.repeat(np.arange(n), np.diff(mat[0])), mat[1] - 1
    m = np.bincount(rows, minlength=n) + np.bincount(cols[rows != cols], minlength=n)
    assert (np.abs(y - z) <= 2 * (m + 1) * 2.0 ** -53 * scale).all()


def test_infinities_stay_where_the_matrix_puts_them():
    """An infinite or NaN x reaches the rows with an entry in its column (a
    stored zero included) and no other."""
    _dev()
    ia, ja, a = _holes(4500, 2)
    a = a.copy()
    a[::11] = 0.0
    n = ia.size - 1
    X = torch.ones(2, n, dtype=torch.float64, device="cuda:0")
    for i, v in ((0, np.inf), (63, -np.inf), (64, np.nan), (2000, np.inf), (n - 1, np.nan)):
        X[:, i] = v
    y, form = _products((ia, ja, a), X, 0)
    z, _ = _products((ia, ja, a), X, 8)
    assert form == -2
    assert np.array_equal(np.isnan(y), np.isnan(z))
    assert np.array_equal(y[np.isinf(z)], z[np.isinf(z)])
    fine = np.isfinite(z)
    assert np.array_equal(fine, np.isfinite(y)) and np.abs(y[fine] - z[fine]).max() < 1e-13


@pytest.mark.parametrize("spmv64", [0, 1])
def test_fp32_inner_solver_on_diagonals(spmv64):
    """The FP32 inner solver reads the diagonal form's FP32 or FP64 values and
    converges to the closed form, whatever the FP32 products' rounding."""
    from jadamilu_amd.jd import Context, lx_optimal
    _dev()
    shape = (23, 21, 19)
    ia, ja, a = M.laplace(shape)
    n = ia.size - 1
    lam, _ = M.laplace_eigs(shape, 3)
    ctx = Context(0)
    ctx.set_option("inner_fp32", 1)
    ctx.set_option("inner_spmv64", spmv64)
    lx = lx_optimal(n, 3, 20)
    X = torch.zeros(lx, dtype=torch.float64, device="cuda:0")
    X[:n] = torch.from_numpy(np.random.default_rng(0).random(n))
    torch.cuda.synchronize()
    r = ctx.pjd(n, a, ja, ia, X.data_ptr(), lx, neig=3, isearch=1, ninit=1, maxiter=4000,
                tol=1e-10, icntl=(0, 1, 0, 0, 1))
    assert r.info == 0 and r.stats["spmv_lanes"] == -2
    np.testing.assert_allclose(r.eigs, lam, rtol=1e-10)
    ctx.close()


def test_other_formats_of_a_matrix_on_diagonals():
    """Option spmv_lanes selects every format on a matrix that took the diagonal
    form, the sliced ELL included, and back."""
    from jadamilu_amd.jd import Context
    _dev()
    n = 67 * 63
    X = torch.randn(2, n, dtype=torch.float64, device="cuda:0")
    ctx = Context(0)
    ctx.set_matrix(*M.laplace((67, 63)))
    results = []
    for lanes in (-2, 0, 4, -2):
        ctx.set_option("spmv_lanes", lanes)
        assert ctx.stats()["spmv_lanes"] == lanes
        Y = torch.zeros(3, n, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ctx.spmv(X.data_ptr(), Y[0].data_ptr())
        ctx.spmm(2, X.data_ptr(), n, Y[1].data_ptr(), n)
        torch.cuda.synchronize()
        results.append(Y)
    ctx.close()
    # five terms a row, of absolute sum 8 max|x| at most, in different orders
    bound = 2 * 6 * 2.0 ** -53 * 8 * float(X.abs().max())
    for Y in results[1:]:
        assert float((Y - results[0]).abs().max()) <= bound
