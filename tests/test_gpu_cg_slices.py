"""CG in one workgroup past the iterations of one launch, on systems that are far from
converged there: a 1D Laplacian with a random right-hand side needs as many iterations as
it has rows.  Residual, direction and solution go through memory between the launches;
a wrong one would show in the history behind 2048 and in the solution.

Tolerances: the kernel and the oracle differ in the order of the dot products alone, the
history is held to the 1e-10 of the other CG tests; two orders of the sums on the CPU
differ by 2e-13 there and by less than 1e-10 in x."""
import numpy as np
import pytest
import torch

import oracle as O
import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu


def laplacian(n):
    cols = np.arange(n)[:, None] + np.array([-1, 0, 1])[None, :]
    ok = (cols >= 0) & (cols < n)
    rowptr = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32)
    vals = np.broadcast_to(np.array([-1.0, 2.0, -1.0]), cols.shape)[ok]
    return P.CSR(n, n, rowptr, cols[ok].astype(np.int32), vals.copy())


@pytest.mark.parametrize("n,kmax", [(4000, 2047), (4000, 2048), (4000, 2049), (4000, 4500),
                                    (4096, 3000), (4096, 4500), (2500, 3000)])
def test_solves_over_several_launches(n, kmax):
    A = laplacian(n)
    oc = O.CSR(n, n, A.rowptr, A.colidx, A.val)
    M = S.Matrix(A.rowptr, A.colidx, A.val, ncols=n)
    b = P.uniform(5, n, -1, 1)
    bd = torch.from_numpy(b).to("cuda:0")
    x, k, hist = S.cg(M, bd, kmax, 1e-10, history=True)
    xo, ko, ho = O.cg(oc, b, kmax, 1e-10)
    assert abs(k - ko) <= 1 and k > 2000
    m = min(k, ko) + 1
    assert np.max(np.abs(np.sqrt(hist[:m] / hist[0]) - np.sqrt(ho[:m] / ho[0]))) <= 1e-10
    if k == ko:
        assert np.linalg.norm(x.cpu().numpy() - xo) <= 1e-10 * np.linalg.norm(xo)
    xn = torch.full((n,), 3.0, dtype=torch.float64, device="cuda:0")
    _, kn, hn = S.cg_noalloc(M, bd, kmax, 1e-10, x=xn, history=True)
    assert kn == k and torch.equal(xn, x) and np.array_equal(hn, hist)
    if kmax > n:
        assert hist[2048] > 1e-8 * hist[0] and hist[k] < 1e-20 * hist[0]
