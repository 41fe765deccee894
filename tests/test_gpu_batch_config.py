"""The block and the lanes of a batched solve are chosen without choosing its teams: the
default rule (4096 rows a member in teams of up to 8) stays until members are named."""
import numpy as np
import pytest

pytest.importorskip("torch")
import torch  # noqa: E402

import spmv_amd as S  # noqa: E402
from spmv_amd import problems as P  # noqa: E402

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def slots(B):
    b = torch.ones((B.nrows, B.nrhs), dtype=torch.float32, device="cuda")
    B.solve(b, max_its=2, rtol=1e-6)
    return B.config()["slots"]


def test_block_and_lanes_leave_the_teams():
    B = S.Batch([P.stencil(5, 200, 250), P.stencil(5, 10, 10)], nrhs=1)  # 50000 rows, 100
    assert slots(B) == 8 + 1
    default = B.config()["rows_per_member"]
    for block, lanes in ((1024, 0), (512, 0), (1024, 2)):
        B.set_config(block, lanes)
        assert slots(B) == 8 + 1, (block, lanes)
        assert B.config()["rows_per_member"] == default
    B.set_config(1024, 0, 4096)  # named: as many as they give
    assert slots(B) == 13 + 1
    assert B.config()["rows_per_member"] == 4096 != default
    B.set_config(1024, 4)
    assert slots(B) == 13 + 1
    B.set_config(1024, 4, default)
    assert slots(B) == 8 + 1
    B.set_config(1024, 4, 0)
    assert slots(B) == 1 + 1
    for bad in (-2, -4096):
        with pytest.raises(S.SpmvError):
            B.set_config(1024, 0, bad)
