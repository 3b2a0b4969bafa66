"""The library's launches, logged on the host (tests/cpp/launch_log.cpp): no GPU."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
PKG = os.path.join(ROOT, "vectorizedadjoint_amd")


def build(directory) -> str:
    exe = str(directory / "launch_log")
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "cpp", "launch_log.cpp"), "-o", exe,
                    "-L", PKG, "-lvectorizedadjoint_amd", "-L", os.path.join(ROCM, "lib"),
                    "-lamdhip64", f"-Wl,-rpath,{PKG}"], check=True)
    return exe


class Launch:
    def __init__(self, line):
        self.recorded = line.startswith("recorded ")
        self.unwritten = "UNWRITTEN" in line
        self.kernel = re.sub(r"^recorded ", "", line).split(" grid=")[0]
        self.fields = dict(re.findall(r"(\w+)=(\S+)", line))

    def __getitem__(self, key):
        return self.fields[key]

    def __repr__(self):
        return f"{self.kernel} {self.fields}"


def log(exe, ops, system, n, np, tableau, batch, adaptive=1, lanes=0, ipw=0, n_obs=0, slots=0,
        flags=0, occupancy=2):
    """One list of launches per op."""
    a = [system, n, np, tableau, adaptive, batch, lanes, ipw, n_obs, slots, flags, occupancy]
    r = subprocess.run([exe, *map(str, a), *ops], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    calls = []
    for line in r.stdout.splitlines():
        if line.startswith("-- "):
            calls.append([])
        elif " grid=" in line:
            calls[-1].append(Launch(line))
    assert len(calls) == len(ops)
    return calls
