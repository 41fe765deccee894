"""csr_wave with complex values, which it runs where every row has a mask over one
list of column offsets: row counts around the 64-row block, widths around its
classes, rows without entries, single and burst stores, results at addresses that
are not 16-byte aligned, ghost columns, the transposed product, new values, and
values that are not finite.  Rows are summed in stored order with separately
rounded operations, so results are compared bit for bit with the oracle."""
import numpy as np
import pytest
import torch

import oracle as O
import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAIR = {"c64": (np.complex128, torch.float64), "c32": (np.complex64, torch.float32)}


def draw(seed, n):
    return P.uniform(seed, n, -1, 1) + 1j * P.uniform(seed + 1, n, -1, 1)


def band(n, offs, keep=None):
    offs = np.asarray(offs, np.int64)
    col = np.arange(n, dtype=np.int64)[:, None] + offs[None, :]
    ok = (col >= 0) & (col < n)
    if keep is not None:
        ok &= keep(col.shape)
    rowptr = np.zeros(n + 1, np.int64)
    np.cumsum(ok.sum(1), out=rowptr[1:])
    return P.CSR(n, n, rowptr.astype(np.int32), col[ok].astype(np.int32), np.ones(int(rowptr[-1])))


def check(A, dtype, wave=True, values=None):
    v = draw(21, A.nnz) if values is None else values
    npt, part = PAIR[dtype]
    x, xt = draw(23, A.ncols).astype(npt), draw(25, A.nrows).astype(npt)
    oc = O.CSR(A.nrows, A.ncols, A.rowptr, A.colidx, A.val)
    want = O.spmv_complex(oc, v.astype(npt), x)
    M = S.Matrix(A.rowptr, A.colidx, v, ncols=A.ncols, dtype=dtype)
    if wave is not None:
        assert ("csr_wave" in M.kernel_name()) == wave, M.kernel_name()
    xd = torch.from_numpy(x).to(DEV)
    # complex entries from the first and from the second element of a buffer: the second
    # is 16-byte aligned for pairs of doubles only
    for off in (0, 1):
        g = torch.full((A.nrows + 3, 2), 7.0, dtype=part, device=DEV)
        y = torch.view_as_complex(g)[off:off + A.nrows]
        M.mult(xd, out=y)
        assert np.array_equal(y.cpu().numpy(), want, equal_nan=True), off
        assert torch.all(g[off + A.nrows:] == 7.0) and torch.all(g[:off] == 7.0)
    if dtype == "c32" or values is not None:
        return M
    yt = M.transpmult(torch.from_numpy(xt).to(DEV)).cpu().numpy()
    assert np.array_equal(yt, O.spmv_t_complex(oc, v, xt))
    v2 = draw(27, A.nnz)
    M.set_values(torch.from_numpy(v2).to(DEV))
    assert np.array_equal(M.mult(xd).cpu().numpy(), O.spmv_complex(oc, v2, x))
    assert np.array_equal(M.transpmult(torch.from_numpy(xt).to(DEV)).cpu().numpy(),
                          O.spmv_t_complex(oc, v2, xt))
    return M


@pytest.mark.parametrize("dtype", ["c64", "c32"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("width", [1, 3, 4, 7, 8, 15, 16, 27])
def test_widths_and_row_counts(dtype, n, width):
    check(band(n, np.arange(width) - width // 2), dtype, wave=None)


@pytest.mark.parametrize("dtype", ["c64", "c32"])
def test_rows_without_entries_and_ghost_columns(dtype):
    rng = np.random.default_rng(4)

    def keep(shape):
        k = rng.random(shape) < 0.85
        k[::71] = False
        k[2500] = True  # the full list
        return k

    check(band(5000, [-900, -30, -1, 0, 1, 30, 900], keep), dtype)
    check(P.stencil(7, 21, 22, 23, ghost_planes=1), dtype)


@pytest.mark.parametrize("dtype", ["c64", "c32"])
def test_burst_stores(dtype):
    """Enough blocks that results are stored in bursts, with a ragged last block."""
    check(P.stencil(7, 111, 101, 97), dtype)


def test_other_matrices_keep_csr_stream():
    check(P.random_spd(5000, 12), "c64", wave=False)
    n, offs = 4133, np.array([-64, -1, 0, 1, 64])  # the first and last rows wrap around
    cols = np.sort((np.arange(n)[:, None] + offs) % n, axis=1)
    check(P.CSR(n, n, (5 * np.arange(n + 1)).astype(np.int32), cols.reshape(-1).astype(np.int32),
                np.ones(5 * n)), "c64", wave=False)


@pytest.mark.parametrize("dtype", ["c64", "c32"])
def test_values_that_are_not_finite(dtype):
    """Infinities and NaN of one row stay in it."""
    A = band(1000, [-30, -1, 0, 1, 30])
    v = draw(21, A.nnz)
    v[A.rowptr[500]:A.rowptr[501]] = complex(np.inf, 1)
    v[A.rowptr[700]] = complex(np.nan, 0)
    check(A, dtype, values=v)
