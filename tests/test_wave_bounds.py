"""Memory bounds of csr_wave, checked without a GPU on what hipcc makes of its parts."""
import os
import re
import shutil
import subprocess

import pytest

from spmv_amd import build as B

pytestmark = pytest.mark.skipif(not (os.path.exists(B.HIPCC) or shutil.which(B.HIPCC)),
                                reason="needs hipcc")


def test_direct_loads_stay_inside_their_range(tmp_path):
    """A buffer load is checked against the buffer's size by its vector and immediate
    offsets; the scalar offset is left out.  So the loads that write LDS have none."""
    src = tmp_path / "fill.hip"
    src.write_text("""
#include "kernels.hpp"
using namespace spmvx;
extern "C" __global__ void fill(const char* g, int32_t bytes, uint32_t* out)
{
  extern __shared__ __align__(16) char buf[];
  lds_fill<5, kLoadStream>(g, bytes, (lds_ptr)buf);
  lds_filled();
  out[threadIdx.x] = reinterpret_cast<const uint32_t*>(buf)[threadIdx.x];
}
""")
    out = tmp_path / "fill.s"
    subprocess.run([B.HIPCC, *B.FLAGS, "--cuda-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    loads = [ln.strip() for ln in out.read_text().splitlines()
             if re.match(r"\s*buffer_load_\S+ .*\blds\b", ln)]
    assert len(loads) == 5
    # vector offset, descriptor, scalar offset; no immediate (it would move the LDS address too)
    for ln in loads:
        assert re.match(r"buffer_load_dwordx4 v\d+, s\[\d+:\d+\], 0 offen( nt)? lds$", ln), ln


def test_burst_stores_read_only_what_is_kept(tmp_path):
    """The lanes of a burst's stores, one after the other on the CPU: the kept results end
    where a page that cannot be read begins, the result vector where one that cannot be
    written does.  Bursts of every length that a plan can choose, whole and ragged last
    blocks, results at and between 16-byte addresses."""
    src = tmp_path / "burst.hip"
    src.write_text("""
#include <sys/mman.h>
#include <cstdio>
#include "kernels.hpp"
using namespace spmvx;

char* guarded_end(size_t bytes) // `bytes` bytes right before a page without access
{
  const size_t whole = (bytes + 4095) / 4096 * 4096;
  char* p = static_cast<char*>(mmap(nullptr, whole + 4096, PROT_READ | PROT_WRITE,
                                    MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
  mprotect(p + whole, 4096, PROT_NONE);
  return p + whole;
}

template <typename X>
int check(const char* name)
{
  const int32_t first = 2, nw = 3, most = 24;
  for (int32_t nkept = 1; nkept <= most; ++nkept)
    for (int32_t cut : {0, 1, 63}) // rows that the last block lacks
      for (int shift : {0, 1})     // elements past a 16-byte address
      {
        const int32_t nrows = (first + (nkept - 1) * nw + 1) * kWaveRows - cut;
        const size_t kb = sizeof(X) * nkept * kWaveRows;
        X* kept = reinterpret_cast<X*>(guarded_end(kb) - kb);
        for (int32_t i = 0; i < nkept * kWaveRows; ++i)
          kept[i] = X(static_cast<float>(i + 1));
        const size_t yb = (sizeof(X) * (nrows + shift) + 15) / 16 * 16;
        X* y = reinterpret_cast<X*>(guarded_end(yb) - yb) + shift;
        std::fprintf(stderr, "%s nkept %d nrows %d shift %d\\n", name, nkept, nrows, shift);
        for (int lane = 0; lane < kWaveRows; ++lane)
          store_burst(kept, nkept, first, nw, nrows, y, lane);
        for (int32_t row = 0; row < nrows; ++row)
        {
          const int32_t b = row / kWaveRows - first, t = b / nw;
          const bool in = b >= 0 && b % nw == 0 && t < nkept;
          const X want = in ? kept[t * kWaveRows + row % kWaveRows] : X(0);
          if (std::memcmp(&y[row], &want, sizeof(X)) != 0)
            return 1;
        }
      }
  return 0;
}

int main()
{
  return check<double>("double") | check<float>("float") | check<cplx<double>>("cplx<double>")
         | check<cplx<float>>("cplx<float>");
}
""")
    exe = tmp_path / "burst"
    subprocess.run([B.HIPCC, *B.FLAGS, "-include", "cstring", "--cuda-host-only", str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr[-200:])
