"""CPU: the captured graphs of the uniform mesh, of one step and of several, with the HIP runtime and the
kernel launches replaced; tests/host/mesh_host_check.cpp."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_graph_bookkeeping(tmp_path):
    exe = str(tmp_path / "mesh_host_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-Wno-unused-result", os.path.join(ROOT, "tests", "host", "mesh_host_check.cpp"),
                           os.path.join(ROOT, "exahype-engine_amd", "csrc", "tables.cpp"), "-o", exe])
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr
