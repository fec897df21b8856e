"""What the host runtime does when the device refuses memory, on the CPU: tests/cpp/host_failures.cpp stands in for HIP,
fails every allocation of a call in turn and checks what the call and the ones after it return."""
import os
import subprocess

import pytest

import vdb_mapping_amd as V

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_failures") / "host_failures")
    lib = os.path.dirname(V.LIB_PATH)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-rdynamic", "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpp", "host_failures.cpp"), "-L" + lib, "-lvdbgpu", "-Wl,-rpath," + lib,
                    "-o", exe], check=True, timeout=300)
    return exe


@pytest.mark.parametrize("scenario", ["snapshot", "section", "update_export", "points"])
def test_refused_memory(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "%s ok" % scenario in r.stdout, r.stdout + r.stderr
