"""csr_wave (one wavefront per 64 rows) at the sizes where it can go wrong: row
counts around the 64-row block, widths around every class, rows with all, some
or none of the column offsets, blocks that fall back to 16-bit indices, few
and many blocks per wavefront (single and burst stores), results at addresses
that are not 16-byte aligned.  Every product sums a row in stored order with
separately rounded operations, so it is compared bit for bit with the oracle
(FP64) and with a 32-bit-index CSR kernel (FP32, BF16)."""
import numpy as np
import pytest
import torch

import oracle as O
import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def from_rows(n, ncols, cols_of, seed):
    """CSR of n rows; cols_of(i) gives row i's ascending columns."""
    rows = [np.asarray(cols_of(i), np.int64) for i in range(n)]
    rowptr = np.zeros(n + 1, np.int64)
    rowptr[1:] = np.cumsum([len(r) for r in rows])
    colidx = np.concatenate(rows + [np.zeros(0, np.int64)])
    return P.CSR(n, ncols, rowptr.astype(np.int32), colidx.astype(np.int32),
                 P.uniform(seed, len(colidx), -1, 1))


def band(n, offs, seed, keep=None):
    """Row i holds columns i + o inside [0, n); keep(rows) masks entries."""
    offs = np.asarray(offs, np.int64)
    col = np.arange(n, dtype=np.int64)[:, None] + offs[None, :]
    ok = (col >= 0) & (col < n)
    if keep is not None:
        ok &= keep(col.shape)
    rowptr = np.zeros(n + 1, np.int64)
    np.cumsum(ok.sum(1), out=rowptr[1:])
    return P.CSR(n, n, rowptr.astype(np.int32), col[ok].astype(np.int32),
                 P.uniform(seed, int(rowptr[-1]), -1, 1))


def check(A, expect_wave=True, masks=None):
    oc = O.CSR(A.nrows, A.ncols, A.rowptr, A.colidx, A.val)
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=A.ncols)
    if expect_wave is not None:
        assert ("csr_wave" in M.kernel_name()) == expect_wave, M.kernel_name()
    if masks is not None:
        assert ("mask" in M.kernel_name()) == masks, M.kernel_name()
    x = P.uniform(77, A.ncols, -1, 1)
    xd = torch.from_numpy(x).to(DEV)
    want = O.spmv(oc, x, threads=8)
    guard = torch.full((A.nrows + 3,), 7.0, dtype=torch.float64, device=DEV)
    for off in (0, 1):  # 16-byte aligned, and not
        y = guard[off:off + A.nrows]
        M.mult(xd, out=y)
        assert np.array_equal(y.cpu().numpy(), want), off
        assert torch.all(guard[off + A.nrows:] == 7.0)
        guard.fill_(7.0)
    for dt, plain in (("f32", 3), ("bf16", 4)):
        L = M.like(dt)
        xf = xd.float()
        g = torch.full((A.nrows + 3,), 7.0, dtype=torch.float32, device=DEV)
        y = L.mult(xf, out=g[1:1 + A.nrows]).clone()
        assert torch.all(g[1 + A.nrows:] == 7.0) and g[0] == 7.0
        y0 = L.mult(xf)
        L.set_kernel(plain)
        ref = L.mult(xf)
        assert torch.equal(y, ref) and torch.equal(y0, ref), dt
    return M


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 511, 1000])
@pytest.mark.parametrize("width", [1, 3, 4, 5, 7, 8, 9, 10, 15, 16, 27])
def test_widths_and_row_counts(n, width):
    """Bands of every class's width and one more, from one row on."""
    lo = width // 2
    check(band(n, np.arange(-lo, width - lo), seed=n * 100 + width), expect_wave=None)


def test_each_class_is_used():
    for width, kr in ((3, 3), (5, 5), (7, 7), (9, 9), (15, 15), (27, 27)):
        M = check(band(3000, np.arange(width) - width // 2, seed=width), masks=True)
        assert f"{kr} column offsets" in M.kernel_name()


def test_subsets_of_the_offsets_and_empty_rows():
    """Rows that use random subsets of 7 spread offsets, some of them none."""
    rng = np.random.default_rng(4)
    offs = [-900, -30, -1, 0, 1, 30, 900]

    def keep(shape):
        k = rng.random(shape) < 0.85
        k[::71] = False
        k[2500] = True  # the full list
        return k

    check(band(5000, offs, 5, keep), masks=True)


@pytest.mark.parametrize("n", [4096, 4133])
def test_blocks_without_masks(n):
    """A periodic operator: the first and last rows wrap around, so their blocks
    keep their 16-bit indices while the others have masks."""
    offs = np.array([-64, -1, 0, 1, 64])
    check(from_rows(n, n, lambda i: np.sort((i + offs) % n), 6), masks=True)


def test_no_masks_one_base_and_windows():
    """Rows alike in length but not in offsets: 16-bit indices for every block,
    from one base and from windows."""
    rng = np.random.default_rng(7)
    A = from_rows(3000, 3000, lambda i: np.sort(rng.choice(np.arange(max(0, i - 400), min(3000, i + 400)), 7, replace=False)), 8)
    assert "one base" in check(A, masks=False).kernel_name()
    n = 200000
    far = 80000

    def cols(i):
        near = rng.choice(np.arange(max(0, i - 300), min(n, i + 300)), 4, replace=False)
        return np.unique(np.concatenate([near, [(i + far) % n, (i + 2 * far) % n]]))

    assert "windows" in check(from_rows(n, n, cols, 9), masks=False).kernel_name()


def test_rows_longer_than_the_gathers_of_a_block():
    """A few rows of 12-30 entries among rows of 7."""
    rng = np.random.default_rng(10)

    def cols(i):
        k = 12 + i % 19 if i % 640 == 5 else 7
        return np.sort(rng.choice(np.arange(max(0, i - 200), min(6400, i + 200)), k, replace=False))

    check(from_rows(6400, 6400, cols, 11), masks=False)


def test_irregular_rows_keep_csr_stream():
    A = P.random_spd(5000, 12)
    check(A, expect_wave=False)


@pytest.mark.parametrize("kind,dims", [(27, (99, 80, 71)), (7, (150, 133, 90)), (5, (1300, 1411, 1))])
def test_burst_stores(kind, dims):
    """Enough blocks that results are stored in bursts, with a ragged last block."""
    check(P.stencil(kind, *dims), masks=True)


def test_rectangular_and_ghost_columns():
    check(P.stencil(27, 21, 22, 23, ghost_planes=1), masks=True)
    # more rows than columns: the last rows hold the last columns
    A = from_rows(1000, 700, lambda i: np.unique(np.clip(i - 150 + np.arange(5), 0, 699)), 13)
    check(A, expect_wave=None)


def test_values_that_are_not_finite():
    """Columns that a row does not have are not read, and values that belong to
    other rows do not enter its sum: infinities and NaN stay where they are."""
    n = 1000
    A = band(n, [-1, 0, 1], 14)
    A.val[A.rowptr[500]:A.rowptr[501]] = np.inf
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=n)
    x = P.uniform(15, n, 0.5, 1)
    x[100] = np.nan
    y = M.mult(torch.from_numpy(x).to(DEV)).cpu().numpy()
    want = O.spmv(O.CSR(n, n, A.rowptr, A.colidx, A.val), x)
    assert np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(y[~np.isnan(y)], want[~np.isnan(want)])
    assert np.isnan(y).sum() == 3 and np.isinf(y).sum() == 1
