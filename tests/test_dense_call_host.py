"""The host side of the dense calls on a stand-in for the HIP runtime (tests/dense_call_host.cpp, CPU):
the record buffer under graph capture, when it grows and when it cannot be allocated; and the LDS that the
fp32-chain kernels ask for against what they read, and the row lengths the MFMA kernels address."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP_INC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists(os.path.join(HIP_INC, "hip", "hip_runtime_api.h")):
        pytest.skip("no g++ or HIP headers")
    out = str(tmp_path_factory.mktemp("dense_call") / "dense_call_host")
    # the host compiler has no __align__ and no HIP_SYMBOL; launchers no scenario reaches stay undefined
    cmd = ["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-D__align__(n)=__attribute__((aligned(n)))",
           "-DHIP_SYMBOL(s)=&s", "-I", HIP_INC, os.path.join(ROOT, "large_model_amd", "csrc", "qmsg_api.cpp"),
           os.path.join(ROOT, "tests", "dense_call_host.cpp"), "-no-pie", "-pthread",
           "-Wl,--unresolved-symbols=ignore-all", "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return out


@pytest.mark.parametrize("scenario", ["capture_small", "capture_large", "no_memory", "no_buffer", "capture_pairs", "few_rows"])
def test_record_buffer(exe, scenario):
    run(exe, scenario)


@pytest.mark.parametrize("scenario", ["chain_lds", "wide_rows", "odd_down"])
def test_kernel_limits(exe, scenario):
    run(exe, scenario)


def run(exe, scenario):
    r = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr[-2000:]
