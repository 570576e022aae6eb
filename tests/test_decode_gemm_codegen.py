"""Code-generation guard for the decode GEMM (csrc/gemm.hip, gemm_kernel).

Its staged instances keep one to three rounds of weights and activations in registers ahead of their use; one round too
many and the allocator spills, which shows in nothing but time. Every instance is compiled for gfx950 with the
library's own flags and must have no scratch (private segment)."""

import os
import re
import shutil
import subprocess
import sys
import tempfile

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "subnetwork-speculative-decoding_amd")


def test_no_instance_spills():
    sys.path.insert(0, PKG)
    import build

    if not os.path.exists(build.HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "gemm.s")
        r = subprocess.run([build.HIPCC, *build.FLAGS, "-I", os.path.join(REPO, "include"), "--offload-device-only", "-S",
                            os.path.join(PKG, "csrc", "gemm.hip"), "-o", out], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        text = open(out).read()
    scratch = {m[1]: int(re.search(r"\.amdhsa_private_segment_fixed_size (\d+)", m[2])[1]) for m in
               re.finditer(r"\.amdhsa_kernel (_ZN3ssd11gemm_kernel\S+)(.*?)\.end_amdhsa_kernel", text, re.S)}
    # 4 row counts x 2 (norm folded or not) x 3 epilogues, for 6 staged (K, tiles) and 13 direct (tiles, waves) plans
    assert len(scratch) == 24 * (6 + 13)
    assert not {k: v for k, v in scratch.items() if v}
