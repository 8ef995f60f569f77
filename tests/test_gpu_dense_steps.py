"""GPU checks of the basis update jdhip_tall_gemm at every number of 4-column
steps of the matrix instruction, with the first and the last number of columns
of each, and at the remainders of its 16-row tiles.

Integer-valued data: every product and partial sum is exact, so the result
equals the host's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _data(n, k):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    A = np.random.default_rng(n + k).integers(-8, 9, (n, k)).astype(float)
    return A, torch.tensor(np.asfortranarray(A).ravel(order="F"), device="cuda:0")


@pytest.mark.parametrize("n,j", [(15, 1), (16, 17), (4097, 10), (140003, 33)])
@pytest.mark.parametrize("k", [k for s in range(1, 17) for k in (4 * s - 3, 4 * s)])
def test_tall_gemm_every_step_count(n, j, k):
    from jadamilu_amd.jd import Context
    V, dV = _data(n, k)
    Q, dQ = _data(k, j)
    dY = torch.full((n * j,), np.nan, dtype=torch.float64, device=dV.device)
    ctx = Context(0)
    ctx.tall_gemm(n, k, j, dV.data_ptr(), n, dQ.data_ptr(), k, dY.data_ptr(), n)
    torch.cuda.synchronize()
    assert np.array_equal(dY.cpu().numpy().reshape(j, n).T, V @ Q)
    ctx.close()
