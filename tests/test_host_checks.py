"""The library's host side over a stub of the HIP runtime (hip_stub.h), which
the check program (host_check.cpp) defines in place of libamdhip64: failing
calls, limited memory and the launches made, without a GPU."""
import os
import shutil
import subprocess

import pytest

from volprim_amd import volprim

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host_check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("host_check") / "host_check")
    lib = os.path.dirname(volprim.LIB_PATH)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-rdynamic",
                    "-o", exe, os.path.join(ROOT, "tests", "host_check.cpp"), f"-L{lib}", "-lvolprim",
                    f"-Wl,-rpath,{lib}", "-Wl,-rpath-link,/opt/rocm/lib", "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("name", ["failed_copies", "export_device", "export_without_memory", "kept_scratch",
                                  "build_memory", "launch_shapes", "batch_images",
                                  "render_beside_server", "path_claims"])
def test_host_check(host_check, name):
    r = subprocess.run([host_check, name], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.startswith(f"ok {name}"), r.stdout + r.stderr
