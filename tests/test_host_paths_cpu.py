"""Host paths of the runtime on a stand-in HIP runtime (host_paths_check.c): with
any one launch or copy of a single-layer call or a prefill failing, the call
returns an error with no work left queued on the caller's memory, and the next
call succeeds; batches of alternating sizes replay no captured step that may hold
a freed buffer."""
import os
import shutil
import subprocess

import pytest

import lpta

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(shutil.which("gcc") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                    reason="gcc or the HIP headers are not available")
def test_host_paths(tmp_path):
    lib = lpta.load_library()._name
    exe = tmp_path / "host_paths_check"
    subprocess.run(["gcc", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-rdynamic", "-o", str(exe),
                    os.path.join(HERE, "host_paths_check.c"), "-I", os.path.join(ROCM, "include"),
                    "-I", os.path.join(os.path.dirname(HERE), "include"), lib, "-Wl,-rpath," + os.path.dirname(lib),
                    "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-Wl,-rpath-link," + os.path.join(ROCM, "lib")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.count(" 0 wrong") == 16
