"""More q-gram list entries than 32 bits count, as the device filter finds them out
(tests/cpu_build/filter_total_cpu.cpp, under AddressSanitizer and UBSan)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_totals_past_32_bits(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "filter_total_cpu"
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=undefined", "-I", str(ROOT / "include"), "-I",
                        str(ROOT / "saruman_amd" / "csrc"),
                        str(ROOT / "tests" / "cpu_build" / "filter_total_cpu.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("OK"), r.stdout + r.stderr
