"""The device memory that the library keeps between calls (csrc/gz_alloc.cpp), as a host program over
a stand-in for the few HIP calls it makes (tests/cpp/test_alloc.cc): no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gizmo_shared_memory_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("alloc") / "test_alloc")
    rocm = os.environ.get("ROCM", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-D__HIP_PLATFORM_AMD__",
                    "-I" + CSRC,
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(rocm, "include"),
                    os.path.join(CSRC, "gz_alloc.cpp"),
                    os.path.join(ROOT, "tests", "cpp", "test_alloc.cc"), "-o", out, "-pthread"],
                   check=True)
    return out


@pytest.mark.parametrize("check", ["refused_wait", "growing_trees", "large_tree", "room_for_others",
                                   "lent_scratch"])
def test_kept_device_memory(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
