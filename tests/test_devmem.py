"""The engine's device memory (csrc/devmem.cpp) on the CPU: against counters in the place of the HIP calls."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "heavyrt_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("devmem") / "devmem_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"), "-I", CSRC, "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "devmem_test.cpp"), os.path.join(CSRC, "devmem.cpp")], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["reuse", "reuse_after_the_sizes_change", "others_get_the_idle_memory",
                                      "not_another_devices", "not_under_capture", "fewer_lanes_without_memory", "threads",
                                      "given_back_at_the_end"])
def test_scenario(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr


def test_every_allocation_can_take_the_idle_memory():
    """hipMalloc and hipMallocAsync themselves are called in devmem.cpp alone."""
    found = []
    for name in sorted(os.listdir(CSRC)):
        if name == "devmem.cpp":
            continue
        with open(os.path.join(CSRC, name)) as fh:
            code = re.sub(r"//[^\n]*", "", fh.read())
        found += [(name, m.group(0)) for m in re.finditer(r"\bhip(Malloc|MallocAsync|MallocManaged|ExtMalloc\w*)\s*\(", code)]
    assert found == []
