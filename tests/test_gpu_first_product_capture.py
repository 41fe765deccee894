"""A matrix's first product captured: whatever its default kernel reads was built with the
matrix.  Replays return what an eager product does, bit for bit."""
import numpy as np
import pytest
import torch

import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16", "c64", "c32"])
@pytest.mark.parametrize("A", [P.random_spd(5000, 12), P.stencil(7, 20, 21, 19)],
                         ids=["irregular", "stencil"])
def test_first_product_captured(A, dtype):
    v = A.val if dtype[0] != "c" else A.val * (1 + 0.5j)
    M = S.Matrix(A.rowptr, A.colidx, v, ncols=A.ncols, dtype=dtype)
    x = torch.from_numpy(P.uniform(3, A.ncols, -1, 1)).to(DEV).to(M.vector_dtype())
    y = torch.empty(A.nrows, dtype=x.dtype, device=DEV)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        M.mult(x, out=y)
    for scale in (1.0, 2.0, -0.5):  # powers of two: exact
        x.mul_(scale)
        y.zero_()
        g.replay()
        assert torch.equal(y, M.mult(x))
        assert torch.isfinite(torch.view_as_real(y) if y.is_complex() else y).all()
