"""The kept device workspace (vt_work.h) on a device of limited memory."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_kept_workspace(tmp_path):
    exe = str(tmp_path / "work")
    b = subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "tests", "cpp", "host_hip"), "-I",
                        os.path.join(ROOT, "voxeltoy_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "work.cpp"),
                        "-o", exe], capture_output=True, text=True)
    assert b.returncode == 0, b.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
