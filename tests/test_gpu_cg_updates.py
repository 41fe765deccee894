"""CG's vector updates with the scalars folded into them and with kernels of their own:
on either side of the number of partial sums that decides, and with the histories.

Three iterations on a 5-point operator against the same three in torch FP64.  FP64
differs in the order of sums: n eps = 5e-10 (2.2e6 rows).  FP32: a sum of n positive
terms in blocks (at most 64 in sequence anywhere, then trees) is within about
64 eps = 8e-6, twice per iteration, three iterations: 5e-5.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import spmv_amd as S  # noqa: E402

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def five_point(nx, ny):
    i = np.arange(nx * ny).reshape(ny, nx)
    pad = np.full((ny + 2, nx + 2), -1)
    pad[1:-1, 1:-1] = i
    cols = np.stack([pad[:-2, 1:-1], pad[1:-1, :-2], i, pad[1:-1, 2:], pad[2:, 1:-1]], -1)
    cols = cols.reshape(-1, 5)
    ok = cols >= 0
    vals = np.broadcast_to(np.array([-1.0, -1.0, 4.5, -1.0, -1.0]), cols.shape)
    rowptr = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32)
    return rowptr, cols[ok].astype(np.int32), np.ascontiguousarray(vals[ok])


def apply(v, nx, ny):
    u = v.view(ny, nx)
    y = 4.5 * u
    y[1:] -= u[:-1]
    y[:-1] -= u[1:]
    y[:, 1:] -= u[:, :-1]
    y[:, :-1] -= u[:, 1:]
    return y.view(-1)


# variant 0 has blocks of at most 256 rows: 4100 partial sums (FP64 apart, FP32
# folded) and 8463 (both apart); the default's are fewer (folded)
@pytest.mark.parametrize("nx,ny", [(1025, 1024), (1473, 1471)])
@pytest.mark.parametrize("variant", [-1, 0])
@pytest.mark.parametrize("dtype,tol", [("f64", 5e-10), ("f32", 5e-5)])
def test_three_iterations(nx, ny, variant, dtype, tol):
    n = nx * ny
    rowptr, colidx, val = five_point(nx, ny)
    A = S.Matrix(rowptr, colidx, val, ncols=n, dtype=dtype)
    A.set_kernel(variant)
    g = torch.Generator(device="cuda").manual_seed(nx)
    b = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) - 0.5
    b = b.to(A.vector_dtype())
    hist = None
    if dtype == "f64":
        x, k, hist = S.cg(A, b, 3, 0.0, history=True)
    else:
        x, k = S.cg_f32(A, b, 3, 0.0)
    assert k == 3
    r = b.double()
    p, want = r.clone(), torch.zeros_like(r)
    norms = [float(r @ r)]
    for _ in range(3):
        y = apply(p, nx, ny)
        a = norms[-1] / (p @ y)
        want += a * p
        r = r - a * y
        norms.append(float(r @ r))
        p = r + (norms[-1] / norms[-2]) * p
    assert torch.linalg.norm(x.double() - want) <= tol * torch.linalg.norm(want)
    if hist is not None:
        np.testing.assert_allclose(np.asarray(hist), norms, rtol=4 * tol)
