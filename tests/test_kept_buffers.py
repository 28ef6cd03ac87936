"""The list of kept device buffers on the CPU: kept_buffers.cpp compiled with
g++ against a recording runtime of two devices (kept_buffers_check.cpp): the
wait for a buffer's own device, the bound of each device, allocations without
room, a refused wait, several threads.  And the likelihood's way of sharing
them with torch: a step that runs out of device memory runs once more after
they have been given back."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_kept_buffers(tmp_path):
    exe = str(tmp_path / "check")
    csrc = os.path.join(ROOT, "hmat-oss_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{csrc}", os.path.join(ROOT, "tests", "kept_buffers_check.cpp"),
                    os.path.join(csrc, "kept_buffers.cpp"), "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_step_without_memory_runs_again(monkeypatch):
    torch = pytest.importorskip("torch")
    gp = pytest.importorskip("hmat_amd.gp")
    calls = []
    monkeypatch.setattr(gp, "release_memory", lambda: calls.append("released"))

    def step(fails):
        calls.append("step")
        if calls.count("step") <= fails:
            raise torch.OutOfMemoryError("no room")
        return 7
    assert gp._with_memory(lambda: step(0)) == 7 and calls == ["step"]
    calls.clear()
    assert gp._with_memory(lambda: step(1)) == 7 and calls == ["step", "released", "step"]
    calls.clear()
    with pytest.raises(torch.OutOfMemoryError):
        gp._with_memory(lambda: step(2))
    assert calls == ["step", "released", "step"]


def test_nothing_kept_nothing_to_release():
    hmat_amd = pytest.importorskip("hmat_amd")
    hmat_amd.release_memory()
