"""Host code of the packed databases on a stand-in for the HIP runtime
(tests/native/fake_hip.h): failed allocations and calls, repeated owners,
devices.  Nothing here needs a GPU."""
import os
import shutil
import subprocess

import pytest

import geneva_amd as G

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    out = str(tmp_path_factory.mktemp("native") / "resident_host")
    lib = os.path.dirname(G.HIP_LIB)
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-rdynamic", "-Wno-unused-result", "-I" + os.path.join(ROOT, "include"),
           "-I/opt/rocm/include", "-o", out, os.path.join(NATIVE, "resident_host_main.cpp"),
           "-L" + lib, "-lgeneva_host", "-lgeneva_hip", "-Wl,-rpath," + lib, "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return out


@pytest.mark.parametrize("case", ["failed_allocation", "no_memory_is_capacity", "owners_twice",
                                  "owners_on_their_device", "packing_fails", "no_host_memory",
                                  "counters_without_slot_engine", "bound_after_huge_estimate",
                                  "refused_turn_is_overflow", "wide_levels_beside_a_large_graph",
                                  "lone_request_does_not_wait", "room_for_tables_set_aside"])
def test_resident_host(exe, case):
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
