"""The pool of device and pinned buffers, built for the CPU on a stand-in for
the runtime that counts allocations, releases and waits."""
import glob
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "baylorlqcd_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pool") / "pool_check")
    subprocess.check_call([os.path.join(ROCM, "llvm", "bin", "clang++"), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                           "-I" + os.path.join(ROCM, "include"), "-I" + CSRC, "-x", "c++",
                           os.path.join(ROOT, "tests", "host", "pool_check.cpp"), os.path.join(CSRC, "qqcd_pool.cpp"),
                           "-o", out])
    return out


@pytest.mark.parametrize("what", ["pinned_wait", "other_size", "pinned_share", "unpooled", "half_built"])
def test_pool(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_every_allocation_can_take_idle_memory():
    """Device memory is asked for through the pool or device_malloc, both of which release idle buffers when the
    card is full."""
    direct = []
    for path in glob.glob(os.path.join(CSRC, "*.cpp")) + glob.glob(os.path.join(CSRC, "*.hip")):
        if os.path.basename(path) == "qqcd_pool.cpp":
            continue
        with open(path) as f:
            code = re.sub(r"//[^\n]*", "", f.read())
        direct += [(os.path.basename(path), m.group(0)) for m in re.finditer(r"\bhip\w*Malloc\w*\s*\(", code)
                   if m.group(0) != "hipHostMalloc("]
    assert not direct
