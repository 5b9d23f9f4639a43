"""The item split's tile ranges (kv_common.h part_range) on the CPU, up to the longest contexts."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CLANG = Path("/opt/rocm/llvm/bin/clang++")


def test_parts_cover_an_item(tmp_path):
    if not CLANG.exists():
        pytest.skip("ROCm clang++ not found")
    out = tmp_path / "item_parts_emu"
    subprocess.run([str(CLANG), "-std=c++17", "-O2", f"-I{ROOT / 'tests' / 'host_emu'}", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'vspec-engine_amd' / 'csrc'}", str(ROOT / "tests" / "host_emu" / "item_parts_emu.cpp"), "-o", str(out)],
                   check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
