"""mlp_dvnd's host logic (csrc/mlp_runtime.cpp) on a HIP runtime of the host
that runs the launches' bookkeeping only (tests/cpp/fake_hip.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "wamca-gpu-mi_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime.h")):
        pytest.skip("no host C++ compiler or HIP headers")
    exe = tmp_path_factory.mktemp("dvnd_host") / "dvnd_host_check"
    src = [os.path.join(ROOT, "tests", "cpp", f) for f in ("dvnd_host_check.cpp", "fake_hip.cpp")]
    subprocess.run(["g++", "-w", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-D__align__(x)=__attribute__((aligned(x)))",
                    "-DHIP_SYMBOL(x)=(&x)", "-I", os.path.join(ROCM, "include"), "-I", CSRC,
                    "-I", os.path.join(ROOT, "include"), *src, os.path.join(CSRC, "mlp_runtime.cpp"), "-pthread",
                    "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("what", ["graphs", "failed_rows", "evaluations", "timed", "fused_grid", "wide_merges"])
def test_dvnd_host(check, what):
    out = subprocess.run([check, what], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
