"""The scratch pools' failure paths, compiled on the host against a HIP runtime
of stubs (tests/c/workspace_check.cpp): no GPU is touched."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failures_leave_no_error_behind(tmp_path):
    exe = tmp_path / "workspace_check"
    csrc = os.path.join(ROOT, "smilei_amd", "csrc")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(rocm, "include"), "-I" + csrc,
                    os.path.join(ROOT, "tests", "c", "workspace_check.cpp"), os.path.join(csrc, "workspace.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, text=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
