"""CG refuses a column map whose halo has another type than the vectors, whatever form its
iterations take, also where the map has no ghosts to fill."""
import numpy as np
import pytest
import torch

import spmv_amd as S
from spmv_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [30, 90, 1200])  # one workgroup, two kernels, three
def test_halo_of_another_type_is_refused(rows):
    A = P.stencil(5, rows, rows)
    m = S.L2GMap(A.nrows)
    M = S.Matrix(A.rowptr, A.colidx, A.val, col_map=m)
    b = torch.ones(A.nrows, dtype=torch.float64, device="cuda:0")
    want, k = S.cg(M, b, 20, 1e-3)
    m.set_halo(np.zeros(0), dtype=S.F32)
    with pytest.raises(S.SpmvError, match="halo dtype differs"):
        S.cg(M, b, 20, 1e-3)
    with pytest.raises(S.SpmvError, match="halo dtype differs"):
        S.cg_noalloc(M, b, 20, 1e-3)
    m.set_halo(np.zeros(0), dtype=S.F64)
    x, k2 = S.cg(M, b, 20, 1e-3)
    assert k2 == k and torch.equal(x, want)
