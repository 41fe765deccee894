"""CG products that keep part of the matrix in the last-level cache: sizes on
either side of the line from which they do, with all and with a part of the blocks kept.

Three iterations on a 7-point operator against the same three in torch FP64.  The
sums differ in order only: n eps = 9e-10 (8e6 rows) bounds their relative error.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import spmv_amd as S  # noqa: E402

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def seven_point(n):
    i = np.arange(n ** 3).reshape(n, n, n)
    cols, vals = [], []
    for axis, sh in ((0, -1), (1, -1), (2, -1), (None, 0), (2, 1), (1, 1), (0, 1)):
        c = i.copy() if axis is None else np.roll(i, -sh, axis)
        if axis is not None:
            edge = [slice(None)] * 3
            edge[axis] = 0 if sh < 0 else -1
            c[tuple(edge)] = -1
        cols.append(c.ravel())
        vals.append(6.5 if axis is None else -1.0)
    cols = np.stack(cols, 1)
    ok = cols >= 0
    rowptr = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32)
    val = np.broadcast_to(np.array(vals), cols.shape)[ok]
    return rowptr, cols[ok].astype(np.int32), np.ascontiguousarray(val)


def apply(v, n):
    u = v.view(n, n, n)
    y = 6.5 * u
    for a in range(3):
        y.narrow(a, 1, n - 1).sub_(u.narrow(a, 0, n - 1))
        y.narrow(a, 0, n - 1).sub_(u.narrow(a, 1, n - 1))
    return y.view(-1)


# 63, 67, 112 (kept whole) and 350 MB of values
@pytest.mark.parametrize("n", [104, 107, 127, 185])
def test_cg_products_with_kept_blocks(n):
    rowptr, colidx, val = seven_point(n)
    A = S.Matrix(rowptr, colidx, val, ncols=n ** 3)
    g = torch.Generator(device="cuda").manual_seed(n)
    b = torch.rand(n ** 3, generator=g, device="cuda", dtype=torch.float64) - 0.5
    x, k = S.cg(A, b, 3, 0.0)
    assert k == 3
    r, p, want = b.clone(), b.clone(), torch.zeros_like(b)
    rr = r @ r
    for _ in range(3):
        y = apply(p, n)
        a = rr / (p @ y)
        want += a * p
        r -= a * y
        new = r @ r
        p = r + (new / rr) * p
        rr = new
    assert torch.linalg.norm(x - want) <= 9e-10 * torch.linalg.norm(want)
