"""The CSR kernel a matrix gets by default, around the lines of its rule: every choice
returns what variant 0 does, bit for bit, as does the transposed product.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import spmv_amd as S  # noqa: E402

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def irregular(n, ncols, mean, seed):
    """1 to 4 * mean entries a row (a few more than a block of 2048), columns anywhere."""
    rng = np.random.default_rng(seed)
    k = rng.integers(1, 2 * mean, n)
    k[:: max(1, n // 3)] = 4 * mean
    if n > 1000:
        k[n // 2] = 2100
    rp = np.concatenate([[0], np.cumsum(k)]).astype(np.int32)
    ci = rng.integers(0, ncols, rp[-1]).astype(np.int32)
    return rp, ci, rng.standard_normal(rp[-1])


# 16-bit columns (ncols <= 65536) and 32-bit; on either side of 2^22 entries
@pytest.mark.parametrize("dtype,want16,want32", [("f64", 9, 4), ("f32", 10, 3), ("bf16", 10, 4)])
@pytest.mark.parametrize("n,mean", [(1, 3), (257, 9), (30000, 20), (200000, 20), (200000, 23)])
def test_default_kernel(dtype, want16, want32, n, mean):
    for ncols in (50000, 300000):
        rp, ci, v = irregular(n, ncols, mean, n + mean)
        M = S.Matrix(rp, ci, v, ncols=ncols, dtype=dtype)
        got = M.kernel()[0]
        if dtype == "f64" and rp[-1] > 1 << 22:
            assert got == (8 if ncols == 50000 else 5)
        elif n > 257:  # (rows of a single block may be alike, or span few columns)
            assert got == (want16 if ncols == 50000 else want32)
        x = torch.rand(ncols, device="cuda", dtype=torch.float64).to(M.vector_dtype())
        xt = torch.rand(n, device="cuda", dtype=torch.float64).to(M.vector_dtype())
        y, yt = M.mult(x), M.transpmult(xt)
        M.set_kernel(0)
        assert torch.equal(y, M.mult(x))
        assert torch.equal(yt, M.transpmult(xt))
        M.set_kernel(-1)
        assert M.kernel()[0] == got
