"""The row kernel's append items (K chunks, V chunks of whole 4-token groups, query chunks)
against the general per-item append, on the CPU with AddressSanitizer: seeded launches over
head dims, block sizes, starts inside a group, packed tokens in and out of order, invalid
table entries, tokens past the table and rotary tables that end inside a group
(tests/host_emu/append_rows_emu.cpp)."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CLANG = Path("/opt/rocm/llvm/bin/clang++")


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    if not CLANG.exists():
        pytest.skip("ROCm clang++ not found")
    out = tmp_path_factory.mktemp("emu") / "append_rows_emu"
    subprocess.run([str(CLANG), "-std=c++17", "-O1", "-g", "-fsanitize=address", "-fno-omit-frame-pointer",
                    f"-I{ROOT / 'tests' / 'host_emu'}", f"-I{ROOT / 'include'}", f"-I{ROOT / 'vspec-engine_amd' / 'csrc'}",
                    str(ROOT / "tests" / "host_emu" / "append_rows_emu.cpp"), "-o", str(out)], check=True,
                   capture_output=True)
    return out


@pytest.mark.parametrize("seed", range(4))
def test_append_rows_equal_general_append(emu, seed):
    r = subprocess.run([str(emu), str(seed), "400"], capture_output=True, text=True,
                       env={"ASAN_OPTIONS": "detect_leaks=0:abort_on_error=0"})
    assert r.returncode == 0, r.stderr[-3000:]


def test_int4_codes_equal_division(tmp_path):
    """int4_nibble against int4_code for every fp16 scale, around each rounding boundary
    (tests/host_emu/int4_codes_emu.cpp)."""
    if not CLANG.exists():
        pytest.skip("ROCm clang++ not found")
    out = tmp_path / "int4_codes_emu"
    subprocess.run([str(CLANG), "-std=c++17", "-O2", "-ffp-contract=off", "-march=native", f"-I{ROOT / 'tests' / 'host_emu'}",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'vspec-engine_amd' / 'csrc'}",
                    str(ROOT / "tests" / "host_emu" / "int4_codes_emu.cpp"), "-o", str(out)], check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
