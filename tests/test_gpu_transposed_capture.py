"""Transposed products captured right after the kernel was changed: whatever the new
kernel of the transposed copy reads was built when it was chosen, not at the first
product.  Replays return what an eager product does, bit for bit."""
import numpy as np
import pytest
import torch

import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype,first,then", [("f64", 3, S.SLICED_VARIANT), ("f64", -1, S.SLICED_VARIANT),
                                              ("f32", 3, S.SLICED_VARIANT), ("f64", 0, -1),
                                              ("c64", -1, 3), ("c64", 3, -1), ("c32", 0, -1)])
def test_captured_after_a_change(dtype, first, then):
    A = P.stencil(7, 30, 31, 29)
    v = A.val if dtype[0] == "f" else A.val * (1 + 0.5j)
    M = S.Matrix(A.rowptr, A.colidx, v, ncols=A.ncols, dtype=dtype)
    x = torch.from_numpy(P.uniform(3, A.nrows, -1, 1)).to(DEV).to(M.vector_dtype())
    y = torch.empty(A.ncols, dtype=x.dtype, device=DEV)
    M.set_kernel(first)
    want = M.transpmult(x).clone()
    M.set_kernel(then)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        M.transpmult(x, out=y)
    for scale in (1.0, 2.0, -0.5):  # powers of two: exact
        x.mul_(scale)
        want = want * scale
        y.zero_()
        g.replay()
        assert torch.equal(y, want)
        assert torch.equal(M.transpmult(x), want)
