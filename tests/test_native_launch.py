"""The launch shapes and tilings of the host plan code on the CPU (no GPU),
built like the plan check of test_native_sanitize.py:
tests/native/launch_check.cpp."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "splinegrids.jl_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def launch_check(tmp_path_factory):
    if not (shutil.which(HIPCC) or os.path.exists(HIPCC)):
        pytest.skip("hipcc not found")
    exe = str(tmp_path_factory.mktemp("launch") / "launch_check")
    cmd = [HIPCC, "-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer", "--offload-arch=gfx950",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-Xarch_host", "-fsanitize=address", "-Xarch_host", "-fsanitize=undefined",
           "-Xarch_host", "-fno-sanitize-recover=all",
           "-x", "hip", "-I", CSRC, os.path.join(CSRC, "sg_plan_host.hip"),
           os.path.join(NATIVE, "launch_check.cpp"), "-o", exe]
    subprocess.run(cmd, check=True, capture_output=True, text=True, timeout=600)
    return exe


@pytest.mark.parametrize("name", ["csr_limit", "csr_many", "groups", "queues",
                                  "gather_lanes", "gradient", "tilings"])
def test_launch_shapes(launch_check, name):
    # the HIP runtime library keeps allocations to the end of the process
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([launch_check, name], capture_output=True, text=True, env=env, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("launch_check ok"), r.stdout + r.stderr
