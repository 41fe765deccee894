"""Calls without a stream run on torch's current one: default, side stream, capture."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import spmv_amd as S  # noqa: E402

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def test_current_stream():
    handle = lambda: S._stream().value or 0  # noqa: E731
    side = torch.cuda.Stream()
    assert handle() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert handle() == side.cuda_stream
    assert (S._stream(side).value or 0) == side.cuda_stream
    assert handle() == torch.cuda.default_stream().cuda_stream


def test_product_in_a_captured_graph():
    n = 1000
    M = S.Matrix(np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32),
                 np.arange(n, dtype=np.float64), ncols=n)
    x = torch.zeros(n, device="cuda", dtype=torch.float64)
    y = torch.empty_like(x)
    M.mult(x, out=y)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        M.mult(x, out=y)
    want = torch.arange(n, device="cuda", dtype=torch.float64)
    for k in (1.0, 2.0, -3.0):
        x.fill_(k)
        graph.replay()
        assert torch.equal(y, k * want)
        torch.cuda.synchronize()
