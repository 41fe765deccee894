"""CG of an indefinite system whose first p.Ap is exactly zero: the step length and the
residual are infinite, not NaN, as in the reference's loop, in every form of the iteration
and whether or not the rows fill the last workgroup."""
import numpy as np
import pytest
import torch

import oracle as O
import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu


# one workgroup with and without idle threads, two kernels, three kernels
@pytest.mark.parametrize("n", [2, 6, 510, 512, 700, 1024, 4094, 4096, 5000, 1100000])
def test_zero_curvature(n):
    val = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
    rowptr, colidx = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    M = S.Matrix(rowptr, colidx, val, ncols=n)
    b = np.ones(n)
    for kmax in (1, 2, 5):
        x, k, hist = S.cg(M, torch.from_numpy(b).to("cuda:0"), kmax, 1e-10, history=True)
        xo, ko, ho = O.cg(O.CSR(n, n, rowptr, colidx, val), b, kmax, 1e-10)
        assert k == ko == kmax
        assert np.array_equal(hist, ho[:kmax + 1], equal_nan=True), (kmax, hist, ho)
        assert np.array_equal(x.cpu().numpy(), xo, equal_nan=True), kmax
    assert np.isinf(hist[1])
