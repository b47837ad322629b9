"""The library's host code against a stand-in of the HIP runtime (CPU, no GPU): memory, streams, failed calls.

The objects of the in-tree build are linked with ``tests/host/runtime_stand_in.cpp`` (device memory is host memory, kernel
launches only count) and the driver ``tests/host/runtime_check.cpp``, whose checks can make an allocation or a launch
fail where a GPU would not on demand.
"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "parallel-in-time-ode-filters_amd" / "csrc"
OBJS = ROOT / "parallel-in-time-ode-filters_amd" / "_build"
SOURCES = ("pof_abi.hip", "pof_inst_d1.hip", "pof_inst_d2.hip", "pof_inst_d3.hip", "pof_inst_d4.hip",
           "pof_registry.hip", "pof_large.hip")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    objs = [OBJS / f"{s}.o" for s in SOURCES]
    cxx = shutil.which("g++")
    if cxx is None or not all(o.exists() for o in objs):
        pytest.skip("g++ or the in-tree build objects are missing (run __graft_entry__.build())")
    exe = tmp_path_factory.mktemp("host") / "runtime_check"
    src = [ROOT / "tests" / "host" / f for f in ("runtime_check.cpp", "runtime_stand_in.cpp")]
    r = subprocess.run([cxx, "-O1", "-g", "-std=c++17", *map(str, src), *map(str, objs), "-lpthread", "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("check", ["kept_memory", "kept_bound", "failed_call", "failed_launch", "failed_upload_of_many",
                                   "captured_stream", "large_shapes"])
def test_runtime_check(driver, check):
    r = subprocess.run([str(driver), check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    assert f"{check}: 0 failures" in r.stdout


def test_every_device_allocation_can_have_the_kept_memory():
    """hipMalloc is called by device_malloc alone."""
    found = []
    for f in sorted(CSRC.iterdir()):
        for n, line in enumerate(f.read_text().splitlines(), 1):
            code = line.split("//")[0]
            if re.search(r"\bhipMalloc(Async|Managed|Pitch)?\s*\(", code) or "hipExtMalloc" in code:
                found.append((f.name, n, code.strip()))
    assert [(f, c) for f, _, c in found] == [("pof_abi.hip", "hipError_t e = hipMalloc(p, bytes);"),
                                             ("pof_abi.hip", "return hipMalloc(p, bytes);")], found
