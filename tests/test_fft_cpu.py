"""The far field's in-place mixed-radix transforms (fft_small.h) run by one CPU thread."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPU = os.path.join(ROOT, "tests", "cpu")


def test_fft_emulation(tmp_path):
    """every length 2^a 3^b 5^c from 8 to 256: the modes against a direct 64-bit DFT, forward then inverse
    against the input, no access outside the sequences.  The error relative to sqrt(n) grows as
    log2(n) times 6e-8: below 1e-6 at 256 points."""
    exe = str(tmp_path / "fft")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wno-unknown-pragmas", "-I" + os.path.join(CPU, "hip_stub"),
                    "-I" + os.path.join(ROOT, "fsd_amd", "csrc"), os.path.join(CPU, "fft_emulation.cpp"), "-o", exe],
                   check=True)
    p = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0, p.stdout
    words = p.stdout.split()
    assert int(words[1]) >= 46 and float(words[-1]) < 1e-6


def test_library_plans_all_or_nothing(tmp_path):
    """the library transforms with any one call of their set-up failing: nothing is left half made; the
    strides of padded rows"""
    exe = str(tmp_path / "lib")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "fsd_amd", "csrc"), os.path.join(CPU, "fft_library_check.cpp"), "-o",
                    exe], check=True)
    p = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0, p.stdout
