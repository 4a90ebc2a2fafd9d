"""The work queue's error word lies in pinned host memory that the host reads while kernels run: every store to it
is at system scope (on gfx950 a store with the sc0 and sc1 bits; an agent-scope one has sc1 alone)."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "g1.cu_amd", "csrc")
SOURCE = """
#include "queue.h"
using namespace g1k;
__global__ void report(int* qerr) { if (threadIdx.x == 0) report_queue_error(qerr, 2); }
__global__ void wait(const unsigned* flag, int* qerr) { wait_flag(flag, 1, qerr, 1); }
"""


def test_error_word_is_stored_at_system_scope(tmp_path):
    if shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    import build
    src, out = tmp_path / "err.hip", tmp_path / "err.s"
    src.write_text(SOURCE)
    subprocess.run(["hipcc", *build.FLAGS, "--cuda-device-only", "-S", "-I", CSRC, str(src), "-o", str(out)], check=True,
                   capture_output=True, timeout=300)
    stores = re.findall(r"^\s*global_store_dword .*$", out.read_text(), re.M)
    assert len(stores) == 2 and all(s.rstrip().endswith("sc0 sc1") for s in stores), stores


def test_error_word_has_one_store():
    """The word's only store in the sources is report_queue_error's."""
    sites = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        for m in re.finditer(r"(?:__hip_atomic_store|__atomic_store\w*|atomic\w+)\s*\(\s*&?(?:\w+(?:\.|->))*qerr\b[^;]*;"
                             r"|\*\s*(?:\w+\.)*qerr\s*=[^=][^;]*;", open(path).read()):
            sites.append((os.path.basename(path), m.group(0)))
    assert sites == [("queue.h", "__hip_atomic_store(qerr, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);")], sites
