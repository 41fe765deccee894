"""CG of small systems (one workgroup; two kernels per iteration) against the
oracle's CG: sizes on both sides of every compiled row count and width and of the
limits of either form, iteration limits around the chunks in which iterations
are launched, a zero right-hand side, and the no-allocation entry point.

Tolerances: the kernels keep the oracle's order of operations on every vector
element and differ in the order of the dot products only.  For these well
conditioned systems (diagonally dominant bands, stencils) the residual history
is held to the 1e-10 of the larger CG tests."""
import numpy as np
import pytest
import torch

import oracle as O
import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def spd_band(n, half, seed):
    """Symmetric band of half-width `half`, strictly diagonally dominant."""
    w = -P.uniform(seed, n * (half + 1), 0.1, 1.0).reshape(half + 1, n)
    cols, vals, rows = [], [], []
    i = np.arange(n)
    for d in range(-half, half + 1):
        j = i + d
        ok = (j >= 0) & (j < n)
        lo = np.minimum(i, j)[ok]
        rows.append(i[ok])
        cols.append(j[ok])
        vals.append(np.zeros(ok.sum()) if d == 0 else w[abs(d), lo])
    rows, cols, vals = map(np.concatenate, (rows, cols, vals))
    order = np.lexsort((cols, rows))
    rows, cols, vals = rows[order], cols[order], vals[order]
    diag = 1.1 * np.bincount(rows, weights=np.abs(vals), minlength=n) + 0.5
    vals = np.where(rows == cols, diag[rows], vals)
    rowptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=rowptr[1:])
    return P.CSR(n, n, rowptr.astype(np.int32), cols.astype(np.int32), vals)


def solve(A, kmax, rtol, b=None):
    oc = O.CSR(A.nrows, A.ncols, A.rowptr, A.colidx, A.val)
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=A.ncols)
    b = P.uniform(91, A.nrows, -1, 1) if b is None else b
    bd = torch.from_numpy(b).to(DEV)
    x, k, hist = S.cg(M, bd, kmax, rtol, history=True)
    x2, k2 = S.cg(M, bd, kmax, rtol)
    assert k2 == k and torch.equal(x, x2)
    xn = torch.full((A.ncols,), 3.0, dtype=torch.float64, device=DEV)
    _, kn, hn = S.cg_noalloc(M, bd, kmax, rtol, x=xn, history=True)
    assert kn == k and torch.equal(xn, x) and np.array_equal(hn, hist)
    xo, ko, ho = O.cg(oc, b, kmax, rtol)
    return x.cpu().numpy(), k, hist, xo, ko, ho


def check(A, kmax=400, rtol=1e-10):
    x, k, hist, xo, ko, ho = solve(A, kmax, rtol)
    assert abs(k - ko) <= 1
    m = min(k, ko) + 1
    assert np.max(np.abs(np.sqrt(hist[:m] / hist[0]) - np.sqrt(ho[:m] / ho[0]))) <= 1e-10
    if k == ko:
        assert np.linalg.norm(x - xo) <= 1e-10 * np.linalg.norm(xo)


@pytest.mark.parametrize("n", [1, 2, 63, 511, 512, 513, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 9000])
def test_row_counts(n):
    check(spd_band(n, 2, n))


# (rows, half-width): rows of 2h + 1 entries on both sides of the widths kept in
# registers for 1, 2, 4 and 8 rows per thread
@pytest.mark.parametrize("n,half", [(300, 3), (300, 13), (300, 14), (300, 27), (300, 28), (900, 4),
                                    (900, 5), (900, 13), (900, 14), (1800, 3), (1800, 6), (1800, 7),
                                    (3000, 1), (3000, 3), (3000, 4), (6000, 1), (6000, 4), (6000, 7),
                                    (6000, 13), (6000, 20), (6000, 31), (6000, 32)])
def test_widths(n, half):
    check(spd_band(n, half, 7 * n + half))


@pytest.mark.parametrize("A", [P.stencil(5, 130, 97), P.stencil(27, 21, 20, 22), P.stencil(7, 40, 41, 39),
                               P.stencil(27, 40, 39, 41), P.stencil(5, 1000, 1049), P.stencil(5, 1000, 1048)],
                         ids=["5pt", "27pt", "7pt", "27pt_large", "rows_over", "rows_in"])
def test_stencils(A):
    check(A, kmax=150, rtol=1e-6)


@pytest.mark.parametrize("n", [700, 5000])
@pytest.mark.parametrize("kmax", [0, 1, 2, 3, 4, 15, 16, 17, 31, 32, 33, 48])
def test_iteration_limits(n, kmax):
    """rtol 0: every solve stops at its limit, with the history up to it."""
    A = P.stencil(5, n // 50, 50)
    x, k, hist, xo, ko, ho = solve(A, kmax, 0.0)
    assert k == ko == kmax and len(hist) == kmax + 1
    assert np.max(np.abs(np.sqrt(hist / hist[0]) - np.sqrt(ho[:kmax + 1] / ho[0]))) <= 1e-10
    assert np.linalg.norm(x - xo) <= 1e-10 * max(np.linalg.norm(xo), 1e-300)


@pytest.mark.parametrize("kmax", [2047, 2048, 2049, 4100])
def test_more_iterations_than_one_launch(kmax):
    """Past convergence the residual stays at rounding level: the solve in one
    workgroup goes on over several launches up to its limit."""
    A = P.stencil(5, 30, 30)
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=A.ncols)
    b = torch.from_numpy(P.uniform(92, A.nrows, -1, 1)).to(DEV)
    x, k, hist = S.cg(M, b, kmax, 1e-290, history=True)
    assert k == kmax or not np.isfinite(hist[k]) or hist[k] == 0.0 or hist[k] / hist[0] < 1e-290 ** 2
    x1, k1, h1 = S.cg(M, b, 150, 0.0, history=True)
    assert np.array_equal(h1, hist[:151])


@pytest.mark.parametrize("n", [700, 5000])
def test_zero_right_hand_side(n):
    """The reference's loop on b = 0: 0/0 in the first iteration, never below the
    tolerance, stops at the limit."""
    A = P.stencil(5, n // 50, 50)
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=A.ncols)
    x, k = S.cg(M, torch.zeros(A.nrows, dtype=torch.float64, device=DEV), 40, 1e-8)
    assert k == 40 and torch.isnan(x).all()


@pytest.mark.parametrize("dims", [(30, 30), (60, 60), (100, 90)])
def test_f32_and_refinement(dims):
    A = P.stencil(5, *dims)
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=A.ncols)
    b = torch.from_numpy(P.uniform(93, A.nrows, -1, 1)).to(DEV)
    oc = O.CSR(A.nrows, A.ncols, A.rowptr, A.colidx, A.val)
    for dt in ("f32", "bf16"):
        L = M.like(dt)
        xl, k = S.cg_f32(L, b.float(), 2000, 1e-4)
        r = O.spmv(oc, xl.double().cpu().numpy()) - b.cpu().numpy()
        assert 0 < k < 2000 and np.linalg.norm(r) <= 2e-4 * np.linalg.norm(b.cpu().numpy())
        x, st = S.ir_cg(M, L, b, rtol=1e-10)
        r = O.spmv(oc, x.cpu().numpy()) - b.cpu().numpy()
        assert st["rel_residual"] <= 1e-10 and np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b.cpu().numpy())


def test_value_updates_and_streams():
    """New values between solves, and a solve on a side stream whose right-hand
    side was written there."""
    A = P.stencil(5, 90, 80)
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=A.ncols)
    b = P.uniform(94, A.nrows, -1, 1)
    for scale in (1.0, 2.0):
        M.set_values(torch.from_numpy(A.val * scale).to(DEV))
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            bd = torch.from_numpy(b).to(DEV) * scale
            x, k = S.cg(M, bd, 500, 1e-10)
        s.synchronize()
        r = O.spmv(O.CSR(A.nrows, A.ncols, A.rowptr, A.colidx, A.val), x.cpu().numpy()) - b
        assert np.linalg.norm(r) <= 1.1e-10 * np.linalg.norm(b)
