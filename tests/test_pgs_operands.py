"""The operands of the four-row PGS blocks (physics.h, pgs_rows and pgs_rows_pair): a block writes the force, the
residuals and the lane mask in its first row and reads the rows' matrix entries up to its last, so no entry may
share a register with a value that the block writes, also where it starts out equal to one. Checked on the
assembly of kernels whose entries are those values."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

SOURCE = """
#include "physics.h"
using namespace g1k;
__global__ void one(float* o, const float* in) {
  const int i = threadIdx.x;
  float A[kMaxEfc] = {}, f = in[i], r = in[64 + i];
  A[0] = in[128 + i]; A[1] = f; A[2] = r; A[3] = in[192 + i];
  unsigned long long lanes = pgs_lanes0();
  pgs_rows<0, 16>(A, i & 15, lanes, f, r);
  o[i] = f; o[64 + i] = r;
}
__global__ void two(float* o, const float* in) {
  const int i = threadIdx.x;
  float A[kMaxEfc] = {}, B[kMaxEfc] = {}, f = in[i], r = in[64 + i], ro = in[128 + i];
  A[0] = in[192 + i]; A[1] = f; A[2] = r; A[3] = ro; B[0] = ro; B[1] = r; B[2] = f; B[3] = A[0];
  unsigned long long lanes = pgs_lanes0();
  pgs_rows_pair<0>(A, B, lanes, f, r, ro);
  o[i] = f; o[64 + i] = r; o[128 + i] = ro;
}
"""


def test_pgs_blocks_keep_their_entries_apart_from_what_they_write(tmp_path):
    if shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    import build
    src, out = tmp_path / "pgs.hip", tmp_path / "pgs.s"
    src.write_text(SOURCE)
    subprocess.run(["hipcc", *build.FLAGS, "--cuda-device-only", "-S", "-I", os.path.join(ROOT, "g1.cu_amd", "csrc"),
                    str(src), "-o", str(out)], check=True, capture_output=True, timeout=300)
    blocks = [b for b in re.findall(r"#ASMSTART(.*?)#ASMEND", out.read_text(), re.S) if "v_fmac_f32_dpp" in b]
    assert [b.count("v_fmac_f32_dpp") for b in blocks] == [4, 8]   # four rows, one or two residuals each
    for b in blocks:
        written = {m for m in re.findall(r"^\s*v_\w+ (v\d+),", b, re.M)}
        entries = re.findall(r"v_fmac_f32_dpp v\d+, v\d+, (v\d+) ", b)
        assert not written & set(entries), b
