"""The library's host code on a stand-in HIP runtime (tests/host_hip): which
kernels a call launches under a device-memory limit, without a GPU."""
import glob
import os
import subprocess

from conftest import ROOT

PKG = os.path.join(ROOT, "chat-wgpu_amd")


def test_prompts_without_room_for_the_batch(tmp_path):
    objs = sorted(glob.glob(os.path.join(PKG, "_build", "*.o")))
    if not objs:
        import build
        build.build()
        objs = sorted(glob.glob(os.path.join(PKG, "_build", "*.o")))
    obj, exe = str(tmp_path / "no_room.o"), str(tmp_path / "no_room")
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    for cmd in ([hipcc, "-std=c++17", "-O1", "-fPIC", "-I", os.path.join(ROOT, "include"), "-c",
                 os.path.join(ROOT, "tests", "host_hip", "no_room.cpp"), "-o", obj],
                ["g++", obj] + objs + ["-lpthread", "-o", exe]):
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
