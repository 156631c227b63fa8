"""What the kernels take for granted of the tables' sizes and of LDS."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = "/opt/rocm/llvm/bin"


def test_table_sizes(tmp_path):
    exe = str(tmp_path / "layout")
    b = subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "voxeltoy_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "layout.cpp"), "-o", exe], capture_output=True, text=True)
    assert b.returncode == 0, b.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout


def test_codes_are_at_the_start_of_lds(tmp_path, vtapi):
    """wf_traverse_kernel without statistics addresses the codes from LDS
    address 0: it may hold no LDS beside the dynamic part."""
    if not os.path.exists(os.path.join(LLVM, "clang-offload-bundler")):
        pytest.skip("no offload bundler")
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    obj = os.path.join(ROOT, "voxeltoy_amd", "_build", "csrc_vt_trace.hip.o")
    if not os.path.exists(obj):
        pytest.skip("the library was built elsewhere")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), "-O", "binary", "--only-section=.hip_fatbin", obj, fat], check=True)
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--type=o", "--unbundle", f"--input={fat}",
                    f"--output={code}", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", code], check=True, capture_output=True, text=True).stdout
    lds = {}
    for k in notes.split("  - .agpr_count")[1:]:
        name = re.search(r"\.name:\s+(\S+)", k.split(".args:")[0] + k[k.rfind(".max_flat_workgroup_size"):])
        size = re.search(r"\.group_segment_fixed_size:\s+(\d+)", k)
        if name and size:
            lds[name.group(1)] = int(size.group(1))
    march = {k: v for k, v in lds.items() if "wf_traverse_kernelILb0E" in k}
    assert len(march) >= 3, sorted(lds)
    assert not any(march.values()), march
