"""A team's wait that runs out ends the batched solve for everyone: members leave their
systems, no further ones are taken, and the call reports it.  The limit is set from the
host (0: the first unsuccessful poll), so every kernel ends as it does in earnest."""
import ctypes
import time

import numpy as np
import pytest

pytest.importorskip("torch")
import torch  # noqa: E402

import spmv_amd as S  # noqa: E402
from spmv_amd import problems as P  # noqa: E402

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("nrhs", [1, 4])
def test_a_wait_that_runs_out_ends_the_solve(monkeypatch, nrhs):
    systems = [P.stencil(5, 150, 200) for _ in range(24)] + [P.stencil(5, 10, 10)]  # 8 members, 1
    ok = S.Batch(systems, nrhs=nrhs)
    monkeypatch.setenv("SPMVX_BATCH_SPIN_LIMIT", "0")
    B = S.Batch(systems, nrhs=nrhs)
    monkeypatch.delenv("SPMVX_BATCH_SPIN_LIMIT")
    b = torch.from_numpy(P.uniform(7, B.nrows * nrhs, -1, 1).astype(np.float32)).cuda()
    b = b.reshape(B.nrows, nrhs)
    x = torch.zeros_like(b)
    for _ in range(2):  # and again: the flag and the queues are reset by every solve
        its = np.full((B.nsys, nrhs), 7, np.int32)
        t0 = time.monotonic()
        rc = S.lib().spmvx_batch_solve(B._h, ctypes.c_void_p(b.data_ptr()),
                                       ctypes.c_void_p(x.data_ptr()), 100000, 1e-30,
                                       its.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(0))
        assert rc != 0
        # 100000 iterations of a system that goes on take a second and more each
        assert time.monotonic() - t0 < 1.0
        assert (its[:24] == -1).any() and np.isin(its[its < 0], [-1]).all()
        with pytest.raises(S.SpmvError, match="timed out"):
            B.solve(b, x, max_its=10, rtol=1e-30)
    xo, io = ok.solve(b, max_its=2000, rtol=1e-4)
    assert (io > 0).all() and torch.isfinite(xo).all()
