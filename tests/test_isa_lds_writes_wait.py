"""A plain s_barrier, unlike __syncthreads(), waits for nothing: a wave that writes LDS for others has to see its writes done
before it passes the next barrier. This test compiles the prompts' kernel to gfx950 ISA and looks, behind every LDS write, for a
wait that covers it before the next barrier.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "effect-torch_amd", "csrc")


def writes_without_a_wait(text):
    """(LDS writes, those that may be under way at the next barrier of the listing), straight-line code between the two."""
    lines = [line.split(";")[0].strip() for line in text.splitlines()]
    writes, open_ones = 0, []
    for i, line in enumerate(lines):
        if not line.startswith("ds_write"):
            continue
        writes += 1
        behind = 0  # LDS instructions behind the write: a count of that many or fewer outstanding leaves the write done
        for follower in lines[i + 1:]:
            if follower.startswith("ds_"):
                behind += 1
            count = re.match(r"s_waitcnt\b.*lgkmcnt\((\d+)\)", follower)
            if count and int(count.group(1)) <= behind:
                break
            if follower.startswith("s_barrier"):
                open_ones.append(i + 1)
                break
            if follower.startswith("s_endpgm"):
                break
    return writes, open_ones


def test_the_detector_sees_the_shape():
    assert writes_without_a_wait("ds_write_b32 v0, v1\ns_waitcnt vmcnt(2)\ns_barrier\n") == (1, [1])
    assert writes_without_a_wait("ds_write_b32 v0, v1\nds_read_b32 v2, v3\ns_waitcnt lgkmcnt(2)\ns_barrier\n") == (1, [1])
    assert writes_without_a_wait("ds_write_b32 v0, v1\nds_read_b32 v2, v3\ns_waitcnt vmcnt(0) lgkmcnt(1)\ns_barrier\n") == (1, [])
    assert writes_without_a_wait("ds_write_b32 v0, v1\ns_waitcnt lgkmcnt(0)\ns_barrier\n") == (1, [])


def test_the_prompts_kernel_waits_for_its_lds_writes(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    out = tmp_path / "gemm_h16_wide.s"
    subprocess.run([hipcc, "-S", "-o", str(out), os.path.join(CSRC, "gemm_h16_wide.hip"), "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "-fPIC", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC,
                    "-I", os.path.join(ROOT, "include"), "--cuda-device-only"],
                   check=True, timeout=900, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    writes, open_ones = writes_without_a_wait(out.read_text())
    assert writes >= 8  # two codecs with minima, waves with and without vectors, last stage and others
    assert open_ones == []
