"""The autotuner's search (autotune.cpp) on the host, with the products it times replaced by a clock."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_search(tmp_path):
    """the fastest shapes are kept, and a product that fails leaves the shapes set before the search"""
    exe = str(tmp_path / "tune")
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "fsd_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpu", "autotune_check.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0, p.stdout
