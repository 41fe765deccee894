"""How a solve decides between its forms, on the CPU: one decision, taken under the
pattern's lock, while another thread is building the pattern's row masks."""
import os
import shutil
import subprocess

import pytest

from spmv_amd import build as B

pytestmark = pytest.mark.skipif(not (os.path.exists(B.HIPCC) or shutil.which(B.HIPCC)),
                                reason="needs hipcc")

SOURCE = """
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include "cg_small.hpp"
using namespace spmvx;

#define EXPECT(c) do { if (!(c)) { std::printf("line %d: %s\\n", __LINE__, #c); return 1; } } while (0)

int main()
{
  Pattern P;
  P.nrows = P.ncols = 64 * 64 * 64;
  P.longest = 27;
  P.nnz = 1900000; // two kernels with masks of 27 offsets, too many entries without
  P.wave = 5;
  EXPECT(!cg_form(P, false).small);
  EXPECT(!cg_form(P, true).small && !cg_form(P, true).tiny);
  const bool room = cg_may_be_small(P);

  // a build in progress: half of what it sets is there
  P.lazy_mu.lock();
  P.masked = true;
  std::atomic<bool> done{false};
  CgForm f;
  std::thread solve([&] {
    f = cg_form(P, true);
    done = true;
  });
  std::this_thread::sleep_for(std::chrono::milliseconds(200));
  const bool early = done;
  P.all_masked = true;
  P.lazy_mu.unlock();
  solve.join();
  EXPECT(!early);
  EXPECT(f.small && f.kr == 27);
  // the workspace is sized alike before and after
  EXPECT(room && cg_may_be_small(P));

  // without masks, and the limits by size
  P.masked = P.all_masked = false;
  P.nnz = 600000;
  EXPECT(cg_form(P, true).small && cg_form(P, true).kr == 0);
  P.nnz = 600001;
  EXPECT(!cg_form(P, true).small);
  P.masked = P.all_masked = true;
  P.wave = 3; // 9 offsets
  P.nnz = 6000000;
  EXPECT(cg_form(P, true).small && cg_form(P, true).kr == 9);
  P.nnz = 6000001;
  EXPECT(!cg_form(P, true).small);
  P.nrows = P.ncols = 4096;
  P.longest = 7;
  EXPECT(cg_form(P, true).tiny && !cg_form(P, true).small);
  P.nrows = P.ncols = (1 << 20) + 1;
  EXPECT(!cg_may_be_small(P) && !cg_form(P, true).small);
  return 0;
}
"""


def test_one_decision_under_the_lock(tmp_path):
    src, exe = tmp_path / "form.hip", tmp_path / "form"
    src.write_text(SOURCE)
    subprocess.run([B.HIPCC, *B.FLAGS, "--cuda-host-only", str(src), "-o", str(exe), "-lpthread"],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
