"""Teams and lanes per row of the batched CG: the edges of both rules.

Each solve ends by the kernel's own check of the true residual in double, so
the residual formed here in double has to meet the tolerance up to the rounding
of 64-bit sums (1e-9 of it allowed); the systems are diagonally dominant, so FP32
CG reaches 1e-5 without exhausting its restarts.
"""
import numpy as np
import pytest

pytest.importorskip("torch")
import torch  # noqa: E402

import spmv_amd as S  # noqa: E402

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


class Banded:
    """n rows, h entries on either side of the diagonal (none wrapped)."""

    def __init__(self, n, h):
        off = np.arange(-h, h + 1)
        cols = np.arange(n)[:, None] + off[None, :]
        ok = (cols >= 0) & (cols < n)
        self.nrows, self.shape = n, (n, n)
        self.rowptr = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32)
        self.colidx = cols[ok].astype(np.int32)
        vals = np.where(off == 0, 2.0 * h + 1.0, -1.0 / (1.0 + np.abs(off)))
        self.val = np.broadcast_to(vals, cols.shape)[ok].astype(np.float32)


def residuals(A, b, x):
    rows = np.repeat(np.arange(A.nrows), np.diff(A.rowptr))
    out = []
    for j in range(b.shape[1]):
        y = np.bincount(rows, A.val.astype(np.float64) * x[A.colidx, j].astype(np.float64),
                        minlength=A.nrows)
        bj = b[:, j].astype(np.float64)
        out.append(np.linalg.norm(bj - y) / np.linalg.norm(bj))
    return np.array(out)


# mean row lengths around the lines of the rule (below 10, up to 32, above), and
# members: one, a remainder, the most of a small team, wide members beyond it
@pytest.mark.parametrize("nrhs", [1, 2, 4])
@pytest.mark.parametrize("h", [0, 1, 4, 5, 15, 16, 40])
@pytest.mark.parametrize("rpm", [None, 300])
def test_lanes_and_small_teams(nrhs, h, rpm):
    systems = [Banded(n, h) for n in (1, 63, 300, 301, 2399, 2401, 4097, 9000)]
    B = S.Batch(systems, nrhs=nrhs)
    if rpm:
        B.set_config(1024, 0, rpm)
    rng = np.random.default_rng(17 * h + nrhs)
    b = rng.uniform(-1, 1, (B.nrows, nrhs)).astype(np.float32)
    for _ in range(3):  # the words of the sums are cleared for every solve
        x, _ = B.solve(torch.from_numpy(b).cuda(), max_its=500, rtol=1e-5)
        xh = x.cpu().numpy()
        for s, A in enumerate(systems):
            lo, hi = B.sys_row[s], B.sys_row[s + 1]
            assert residuals(A, b[lo:hi], xh[lo:hi]).max() <= 1e-5 * (1 + 1e-9), (s, h, nrhs)


@pytest.mark.parametrize("rows", [131072, 131073, 160001])
def test_wide_members_beyond_a_small_team(rows):
    systems = [Banded(rows, 2), Banded(50, 2)]
    B = S.Batch(systems, nrhs=4)
    b = np.random.default_rng(5).uniform(-1, 1, (B.nrows, 4)).astype(np.float32)
    x, _ = B.solve(torch.from_numpy(b).cuda(), max_its=500, rtol=1e-5)
    assert residuals(systems[0], b[:rows], x.cpu().numpy()[:rows]).max() <= 1e-5 * (1 + 1e-9)
    assert B.config()["slots"] == max(8, -(-rows // 16384)) + 1


@pytest.mark.parametrize("rows", [40000, 131073])
def test_chosen_members_are_not_widened(rows):
    """Rows per member set by the caller: teams of as many members as they give, up to a
    sixteenth of the CUs (one workgroup of 1024 threads each)."""
    systems = [Banded(rows, 2), Banded(50, 2)]
    B = S.Batch(systems, nrhs=4)
    B.set_config(1024, 0, 4096)
    b = np.random.default_rng(6).uniform(-1, 1, (B.nrows, 4)).astype(np.float32)
    x, _ = B.solve(torch.from_numpy(b).cuda(), max_its=500, rtol=1e-5)
    assert residuals(systems[0], b[:rows], x.cpu().numpy()[:rows]).max() <= 1e-5 * (1 + 1e-9)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert B.config()["slots"] == min(cus // 16, -(-rows // 4096)) + 1
