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
