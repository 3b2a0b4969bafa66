"""The checkpoint spacings of observed solves, CPU only: obs_stride_max and
obs_first_stride (vectorizedadjoint_amd/csrc/va_kernels.hpp) followed through a
forward on the host for every cap, slot count and pair of step counts of two solves.
A solve that starts from the spacing of one that took all of its steps (count = cap)
must not start above the spacing that the reverse's row buffers are sized for: with
slots * stride_max == cap it did, and segments of twice the rows were written."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_segments_fit_the_row_buffers(tmp_path):
    exe = str(tmp_path / "obs_stride_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(ROOT, "vectorizedadjoint_amd", "csrc"), "-I",
                    os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "cpp", "obs_stride_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe, "80"], capture_output=True, text=True, check=True)
    checked, bad = r.stdout.split()[-3], r.stdout.split()[-1]
    assert int(checked) > 3_000_000 and int(bad) == 0, r.stdout
