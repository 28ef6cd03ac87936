"""The list of kept device buffers on the CPU: kept_buffers.cpp compiled with
g++ against a recording runtime of two devices (kept_buffers_check.cpp): the
wait for a buffer's own device, the bound of each device, allocations without
room, a refused wait, several threads."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_kept_buffers(tmp_path):
    exe = str(tmp_path / "check")
    csrc = os.path.join(ROOT, "hmat-oss_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{csrc}", os.path.join(ROOT, "tests", "kept_buffers_check.cpp"),
                    os.path.join(csrc, "kept_buffers.cpp"), "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
