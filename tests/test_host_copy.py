"""The threads of a large host copy (csrc/host_copy.hpp): no more than the cores
that the process may run on leave beside the caller's, and eight at most."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
PROGRAM = """
#include <cstdio>
#include "host_copy.hpp"
int main() { printf("%d", hostcopy::workers()); }
"""


@pytest.mark.skipif(not os.path.isdir(os.path.join(HIP, "hip")), reason="no HIP headers")
def test_workers_follow_the_allowed_cores(tmp_path):
    src, exe = tmp_path / "workers.cpp", tmp_path / "workers"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", HIP, "-I",
                    os.path.join(ROOT, "cps_veloc_amd", "csrc"), str(src), "-o", str(exe),
                    "-pthread"], check=True, capture_output=True)
    cores = sorted(os.sched_getaffinity(0))
    for n in sorted({1, 2, 3, len(cores)} & set(range(len(cores) + 1))):
        out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=20,
                             preexec_fn=lambda: os.sched_setaffinity(0, cores[:n])).stdout
        assert int(out) == min(8, n - 1)
