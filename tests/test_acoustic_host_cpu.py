"""CPU: the host logic of the acoustic mesh (steps, gradient, their buffers) on a
device made of host memory that can run out; tests/host/acoustic_host_check.cpp."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


SCENARIOS = ["dataflow", "stale_error", "failed_allocation", "no_second_faces", "gradient_without_room", "many_meshes",
             "large_mesh", "threads"]


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "acoustic_host_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-Wno-unused-result", os.path.join(ROOT, "tests", "host", "acoustic_host_check.cpp"),
                           os.path.join(ROOT, "exahype-engine_amd", "csrc", "tables.cpp"), "-pthread", "-o", exe])
    return exe


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_scenario(check, scenario):
    p = subprocess.run([check, scenario], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr
