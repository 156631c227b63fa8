"""The staging ring of vt_staging.h on the CPU, with a device of one thread in
place of the runtime (tests/cpp/staging_runtime.h)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/llvm/bin/clang++"
INCLUDES = [f"-I{os.path.join(ROOT, p)}" for p in ("tests/cpp/host_hip", "tests/cpp", "voxeltoy_amd/csrc")]


def run(tmp_path, source, *args, cxx="g++", flags=()):
    exe = str(tmp_path / source.split(".")[0])
    b = subprocess.run([cxx, "-O2", "-std=c++17", "-pthread", *flags, *INCLUDES,
                        os.path.join(ROOT, "tests", "cpp", source), "-o", exe], capture_output=True, text=True)
    assert b.returncode == 0, b.stderr
    return subprocess.run([exe, *args], capture_output=True, text=True, timeout=100)


def test_workers_leave_a_copy_that_ended(tmp_path):
    r = run(tmp_path, "staging_order.cpp", "1500")
    assert r.returncode == 0, r.stdout + r.stderr
    assert "late looks 0 wrong bytes 0" in r.stdout


@pytest.mark.skipif(not os.path.exists(CLANG), reason="ROCm clang not present")
def test_ring_has_no_data_race(tmp_path):
    r = run(tmp_path, "staging_order.cpp", "120", cxx=CLANG, flags=("-g", "-fsanitize=thread"))
    assert "ThreadSanitizer" not in r.stderr, r.stderr[-4000:]
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]


def test_copy_behind_a_long_kernel_sleeps_and_leaves_the_ring(tmp_path):
    r = run(tmp_path, "staging_busy.cpp")
    assert r.returncode == 0, r.stdout + r.stderr


def test_one_small_copy_makes_no_ring(tmp_path):
    r = run(tmp_path, "staging_first.cpp")
    assert r.returncode == 0, r.stdout + r.stderr
