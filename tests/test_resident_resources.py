"""The resident kernels' resources, from the compiler's report that build() records beside the library: two
waves per SIMD without scratch, which the batch sizes they take (launch_form) count on."""
import json
import os

import pytest

from conftest import ROOT


def test_resident_kernels_keep_two_waves_per_simd():
    path = os.path.join(ROOT, "g1.cu_amd", "build", "resource_usage.json")
    if not os.path.exists(path):
        pytest.skip("no resource report (run __graft_entry__.build())")
    res = {f: r for f, r in json.load(open(path)).items() if "k_resident" in f}
    assert len(res) == 4, list(res)
    for fn, r in res.items():
        assert r["Occupancy"] >= 2 and r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0, (fn, r)
        assert r["VGPRs"] + r["AGPRs"] <= 256, (fn, r)
        # 1024 two-wave blocks (one world each) or 2048 one-wave blocks at once: 4 or 8 per CU of 160 KB LDS
        assert r["LDS Size"] <= (160 * 1024) // (4 if "ILb1E" in fn else 8), (fn, r)
