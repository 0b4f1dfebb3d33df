"""The engine at the limit of its device memory, and which kernels it launches: each scenario in a process of its own,
where tests/cpp/hip_shim.c stands in front of the HIP calls."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT
from gpu_util import say

pytestmark = pytest.mark.gpu

WORKER = os.path.join(ROOT, "tests", "gpu_memory_worker.py")


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("shim") / "hip_shim.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", "-o", lib, os.path.join(ROOT, "tests", "cpp", "hip_shim.c"),
                    "-ldl", "-lpthread"], check=True)
    return lib


@pytest.mark.parametrize("scenario", ["idle_memory", "smaller_launches", "refused_refit", "wide_nodes", "candidates"])
def test_scenario(gpu_ctx, shim, scenario):
    say(f"memory: {scenario}")
    r = subprocess.run([sys.executable, WORKER, shim, scenario], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and f"done {scenario}" in r.stdout, r.stdout + r.stderr
