"""The device filter's packed-code helpers, compiled for the host under ASan and
UBSan, against a byte-by-byte reading of the same bases."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_packed_codes_equal_bytes(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "filter_packed_cpu"
    cmd = [gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
           "-fno-sanitize-recover=undefined", "-I", str(ROOT / "include"),
           "-I", str(ROOT / "saruman_amd" / "csrc"),
           str(ROOT / "tests" / "cpu_build" / "filter_packed_cpu.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("OK"), r.stdout + r.stderr
