"""The host engine (sapporo2_amd/csrc/engine.cpp) on the CPU, against a HIP runtime of the
test's own whose queue runs as late as the engine's waits allow (tests/native/fake_hip.h):
memory reused before the device has read it, calls that fail half way, and what the engine
asks of the kernels."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")
CSRC = os.path.join(ROOT, "sapporo2_amd", "csrc")
HIP_INC = "/opt/rocm/include"


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(HIP_INC):
        pytest.skip("g++ or the HIP headers not available")
    exe = str(tmp_path_factory.mktemp("engine") / "engine_check")
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-fsanitize=undefined", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
           "-I", HIP_INC, "-I", CSRC, "-I", NATIVE, os.path.join(NATIVE, "engine_check.cpp"),
           os.path.join(CSRC, "engine.cpp"), "-o", exe, "-pthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("check", ["failed_calls", "failed_growth", "send_release", "failed_send", "load_capacity", "xcd_shapes",
                                   "noalloc_shapes", "pick_up", "scratch_size", "mode_shapes",
                                   "batch_range"])
def test_engine(harness, check):
    env = dict(os.environ, SAPPORO2_AMD_HOST_THREADS="4")
    r = subprocess.run([harness, check], capture_output=True, text=True, env=env, timeout=300)
    assert r.returncode == 0 and "ok" in r.stdout, (r.stdout + r.stderr)[-4000:]
    assert "runtime error" not in r.stderr, r.stderr[-4000:]
