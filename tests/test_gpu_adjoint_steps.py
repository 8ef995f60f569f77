"""The gradient kernels at every number of vectors where the count of loads in
flight changes, on rows of 0 to 9 entries and at the limits of row length and
entries of a wave, against the formula in NumPy.

Both sides form the same products in double, at most 64 of them in a sum: they
agree to 64 * 2^-52 of the sum of absolute terms.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _check(rows, n, k, rng):
    """Both gradients for the rows' columns (0-based, upper triangle)."""
    from jadamilu_amd import lib
    ia = np.concatenate([[1], 1 + np.cumsum([r.size for r in rows])]).astype(np.int32)
    ja = (np.concatenate(rows) + 1).astype(np.int32)
    ldx = n + 3
    X, w = rng.standard_normal((k, ldx)), rng.standard_normal(k)
    dev = [torch.from_numpy(v).cuda() for v in (ia, ja, X)]
    g = torch.full((ja.size,), np.nan, dtype=torch.float64, device="cuda:0")
    d = torch.full((n,), np.nan, dtype=torch.float64, device="cuda:0")
    wp = w.ctypes.data_as(C.POINTER(C.c_double))
    torch.cuda.synchronize()
    assert lib().jdhip_adjoint_csr(None, n, dev[0].data_ptr(), dev[1].data_ptr(),
                                   dev[2].data_ptr(), ldx, k, wp, g.data_ptr()) == 0
    assert lib().jdhip_adjoint_diag(None, n, dev[2].data_ptr(), ldx, k, wp, d.data_ptr()) == 0
    torch.cuda.synchronize()
    i, j = np.repeat(np.arange(n), np.diff(ia)), ja - 1
    c = np.where(i == j, 1.0, 2.0)
    t = w[:, None] * X[:, i] * X[:, j]
    assert (np.abs(g.cpu().numpy() - c * t.sum(0)) <= 64 * 2.0 ** -52 * c * np.abs(t).sum(0)).all()
    t = w[:, None] * X[:, :n] ** 2
    assert (np.abs(d.cpu().numpy() - t.sum(0)) <= 64 * 2.0 ** -52 * np.abs(t).sum(0)).all()


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 9, 10, 11, 12, 13, 16, 17, 33, 64])
@pytest.mark.parametrize("n", [1, 63, 65, 1500, 32767, 32768 + 65])
def test_gradients_at_every_step(n, k):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    rng = np.random.default_rng(n + k)
    rows = [np.unique(np.append(rng.integers(i, n, i % 9), i)) if i % 7 else np.array([], int)
            for i in range(n)]
    rows[n - 1] = np.array([n - 1])
    _check(rows, n, k, rng)


# Row lengths of 64 rows at the limits up to which a wave gives each lane a row (16
# entries a row, 512 in its 64 rows): all at a limit, one entry over it, a long
# row among short ones; beside waves that decide otherwise and as a last wave of
# few rows.  Matrices of at least 32,768 rows have such waves.
LENGTHS = {
    "row 16": [16] + [0] * 63, "row 17": [17] + [0] * 63,
    "wave 512": [8] * 64, "wave 513": [8] * 63 + [9],
    "wave 512 of 16": [16] * 32 + [0] * 32, "wave 513 of 16": [16] * 32 + [1] + [0] * 31,
    "long row": [3] * 40 + [150] + [0] * 23, "empty": [0] * 64,
}


@pytest.mark.parametrize("k", [1, 3, 10, 16])
@pytest.mark.parametrize("name", list(LENGTHS))
@pytest.mark.parametrize("tail", [1, 41])
def test_gradients_at_the_limits_of_a_wave(name, tail, k):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    lengths = [1] * 32768 + [5] * 64 + LENGTHS[name] + [12] * 64 + LENGTHS[name][-tail:]
    n = len(lengths)
    rng = np.random.default_rng(k)
    # (any columns: the kernel does not ask for the upper triangle)
    _check([np.array([i]) if i < 32768 else np.sort(rng.choice(n, m, replace=False))
            for i, m in enumerate(lengths)], n, k, rng)
