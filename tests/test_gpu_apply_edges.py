"""The preconditioner apply's kernels at the sizes where they can go wrong,
against the oracle's apply on the same factor.

Tolerance: both sides sum the same products in double in another order; the
existing parity bar of the FP64 apply (1e-12 relative) holds throughout.
"""
import numpy as np
import pytest

from jadamilu_amd import matrices as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _hub(n, k):
    """A path of n nodes and a hub coupled to the last k of them (SPD): the
    coupling block holds a row of about k entries."""
    r = np.arange(n - 1)
    c = np.arange(n - k, n)
    diag = np.full(n + 1, 4.0)
    diag[-1] = 2.0 * n
    rows, cols = np.concatenate([r, c]), np.concatenate([r + 1, np.full(k, n)])
    return M.from_pairs(n + 1, rows, cols, -np.ones(rows.size), diag)


def _check(gen, options, sweeps, coupling=0, single=False, spd=True, dense_max=300):
    """The apply against the oracle's; the factor, the kernel forms chosen and
    the bytes that a forward sweep of the first level is said to take."""
    from jadamilu_amd.ildl import IldlFactor
    from jadamilu_amd.jd import Context
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    ia, ja, a = gen()
    n = ia.size - 1
    f = IldlFactor(n, ia, ja, a, droptol=1e-3, spd=spd, single=single, dense_max=dense_max,
                   coupling=coupling)
    assert f.ierr == 0
    ctx = Context(0)
    for name, value in options.items():
        ctx.set_option(name, value)
    ctx.attach_ildl(f, sweeps=sweeps)
    ex = f.export()
    rng = np.random.default_rng(3)
    for _ in range(2):
        r = rng.standard_normal(n)
        rd = torch.tensor(r, device="cuda:0")
        zd = torch.full_like(rd, float("nan"))
        torch.cuda.synchronize()
        ctx.precond_apply(zd.data_ptr(), rd.data_ptr())
        torch.cuda.synchronize()
        zo = O.ildl_apply(ex, r, sweeps=sweeps)
        tol = 2e-5 if single else 1e-12
        assert np.linalg.norm(zd.cpu().numpy() - zo) <= tol * np.linalg.norm(zo)
    forms, nbytes = ctx.ildl_level_forms(), ctx.ildl_time_sweep(1)[1]
    ctx.close()
    return ex, forms, nbytes


def _stream_bytes(level, value, vector):
    """What a forward sweep in the CSR-stream form reads and writes when the
    factor's own order is kept, and its entries by the width of their columns:
    blocks of up to 256 rows and 512 entries (1024 from 800,000 on); 16-bit
    columns where a block spans less than 65,536 of them, if seven eighths of
    the blocks do.  value, vector: bytes of an entry and of a vector's."""
    ptr, idx = level["lb_ptr"].astype(np.int64), level["lb_idx"]
    n, nnz = ptr.size - 1, int(ptr[-1])
    cap = 1024 if nnz >= 800000 else 512
    assert np.diff(ptr).max() <= cap
    r, nblk, wide_blocks, narrow, wide = 0, 0, 0, 0, 0
    while r < n:
        r0 = r
        r = min(n, r0 + 256, int(np.searchsorted(ptr, ptr[r0] + cap, "right")) - 1)
        cols = idx[ptr[r0]:ptr[r]]
        nblk += 1
        if cols.size and int(cols.max()) - int(cols.min()) >= 65536:
            wide += cols.size
            wide_blocks += 1
        else:
            narrow += cols.size
    if 8 * wide_blocks > nblk:
        narrow, wide = 0, wide + narrow
    total = value * nnz + 2 * narrow + 4 * wide + 2 * (n + nblk) + 20 * nblk + 3 * vector * n
    return total, narrow, wide


# rows around the 512 entries that a block of the small CSR-stream form holds
@pytest.mark.parametrize("k", [508, 509, 510, 511, 512, 513])
@pytest.mark.parametrize("single", [False, True])
def test_stream_rows_at_the_block_size(k, single):
    _check(lambda: _hub(700, k), {"ildl_form": 1}, 3, single=single)


# a row of k - 1 entries of L_B, or (k = 4000) of 1,281 of the coupling block,
# among rows of one: lane groups up to 16 times their 8 lanes, CSR-stream beyond;
# forms of the forward and backward sweeps and of the coupling block
@pytest.mark.parametrize("k,form", [(100, [8, 8]), (129, [8, 8]), (130, [1, 8]),
                                    (4000, [8, 8, 1])])
def test_long_row_among_short_ones(k, form):
    _, forms, _ = _check(lambda: _hub(4000, k), {}, 3, dense_max=0)
    assert forms[0][:len(form)] == form


# one, two and three sweeps: where the last sweep carries D^-1 and the addition
# of the second solve, with 1x1 and with 2x2 pivots, in every family of forms,
# replayed and launched one by one
@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("coupling", [0, 1])
@pytest.mark.parametrize("form", [0, 1, 8])
@pytest.mark.parametrize("sweeps", [1, 2, 3])
@pytest.mark.parametrize("gen,spd", [(lambda: M.laplace((13, 11, 9)), True),
                                     (lambda: M.anderson(11, 16.5, 4), False)])
def test_fused_ends_of_the_sweeps(gen, spd, sweeps, form, coupling, graph):
    for single in (False, True):
        _check(gen, {"ildl_form": form, "ildl_graph": graph}, sweeps, coupling=coupling,
               single=single, spd=spd, dense_max=50)


# the column widths of the CSR-stream form, 16 bits, some blocks in 32 and all in
# 32, at both block sizes; the bytes that the sweep reports say which was taken
@pytest.mark.parametrize("gen,spd,widths", [
    (lambda: M.laplace((30, 29, 28)), True, (True, False)),
    (lambda: M.laplace((46, 45, 44)), True, (True, True)),
    (lambda: M.laplace((48, 46, 44)), True, (False, True)),
    (lambda: M.anderson(42, 16.5, 1), False, (True, False)),
    (lambda: M.anderson(44, 16.5, 1), False, (True, True)),
    (lambda: M.laplace((62, 61, 60)), True, (False, True)),
])
@pytest.mark.parametrize("single", [False, True])
def test_stream_column_widths(gen, spd, widths, single):
    ex, _, nbytes = _check(gen, {"ildl_form": 1, "ildl_storage": 0}, 2, single=single, spd=spd)
    total, narrow, wide = _stream_bytes(ex["levels"][0], 4 if single else 8,
                                        4 if single and spd else 8)
    assert (narrow > 0, wide > 0) == widths
    assert nbytes == total


# a level large enough for the blocks of 1024 entries
def test_stream_wide_blocks():
    _check(lambda: M.laplace((64, 63, 61)), {"ildl_form": 1}, 2)


def test_stream_long_row_among_wide_blocks():
    """A coupling block of more than 800,000 entries, so in blocks of 1024, with
    a row of some thousand entries."""
    def gen():
        parts = [M.laplace((86, 85, 84)), _hub(30000, 30000)]
        n = parts[0][0].size - 1
        return (np.concatenate([parts[0][0][:-1], parts[1][0] + parts[0][0][-1] - 1]),
                np.concatenate([parts[0][1], parts[1][1] + n]),
                np.concatenate([p[2] for p in parts]))
    ex, _, _ = _check(gen, {"ildl_form": 1}, 2)
    ptr = ex["levels"][0]["lc_ptr"]
    assert ptr[-1] >= 800000 and np.diff(ptr).max() > 1024


def test_apply_on_a_stream_under_capture():
    """A replayed apply launches kernel by kernel while its stream is captured
    (a graph launch cannot be), and the captured graph gives the same values
    on every replay, with the context's own replays between them."""
    from jadamilu_amd.ildl import IldlFactor
    from jadamilu_amd.jd import Context
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    ia, ja, a = M.laplace((20, 19, 18))
    n = ia.size - 1
    ctx = Context(0)
    ctx.attach_ildl(IldlFactor(n, ia, ja, a, droptol=1e-3, spd=True, dense_max=100), sweeps=3)
    r = torch.rand(n, dtype=torch.float64, device="cuda:0")
    z, zc = torch.zeros_like(r), torch.zeros_like(r)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.ExternalStream(ctx.stream_ptr()),
                          capture_error_mode="thread_local"):
        ctx.precond_apply(zc.data_ptr(), r.data_ptr())
    for _ in range(4):
        r.uniform_(-1.0, 1.0)
        zc.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ctx.precond_apply(z.data_ptr(), r.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(z, zc) and float(z.abs().max()) > 0.0
    ctx.close()
