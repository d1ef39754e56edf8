"""The host side of the C ABI (psp_amd/csrc/psp_hip.cpp) without a GPU, by
tests/host_driver_check.cpp: built here with the address and undefined sanitizers
against a HIP runtime of host memory, whose kernels compute nothing and check
that their arrays are live and large enough.  Which calls factor and allocate
when the fused launches are switched on after Initialize, with the memory for
their layout and without it; Initialize after one that ran out of memory at any
of its allocations; the memory that Initialize takes at most, no more than the
factors twice with the scratch of their updates and inverses; and several
factored contexts, whose factorizations share an array."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "psp_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "host_driver_check")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-D__HIP_PLATFORM_AMD__", "-D__align__(x)=",
                    "-DHIP_SYMBOL(x)=((const void*)&x)", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(ROOT, "tests", "host_driver_check.cpp"),
                    os.path.join(CSRC, "psp_hip.cpp"), os.path.join(CSRC, "symbolic.cpp"),
                    "-o", exe], check=True)
    return exe


# mode nx ny nz [precision]
@pytest.mark.parametrize("args", [
    "fused 24 22 30", "fused 40 40 24 1", "oom 24 22 30", "oom 24 22 30 1", "retry 14 13 24",
    "retry 9 13 27 1", "memory 100 100 100", "memory 144 128 80", "memory 200 200 100 1",
    "several 24 22 30", "several 61 47 83 1",
])
def test_host_driver(checker, args):
    out = subprocess.run([checker] + args.split(), capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, (out.stdout + out.stderr)[-3000:]
