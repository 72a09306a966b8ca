"""The context's growable buffers (csrc/dev_buf.h) on a runtime that counts
allocations: a block that a captured call was bound to outlives growth."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_dev_buf(tmp_path):
    exe = tmp_path / "dev_buf_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__",
                    "-Xlinker", "--no-undefined", "-I", "/opt/rocm/include",
                    "-I", os.path.join(ROOT, "vkqlora.rs_amd", "csrc"),
                    os.path.join(ROOT, "tests", "dev_buf_check.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "failures=0" in r.stdout, r.stdout
