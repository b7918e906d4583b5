"""The device filter's pairing with a read's lists staged, as its kernel holds them in
LDS, whole or cut short: the host filter's candidates, batches and perfect hits
(tests/cpu_build/filter_staged_cpu.cpp, under AddressSanitizer and UBSan)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    from saruman_amd import _build
    if not _build.LIB.exists():
        pytest.skip("libsaruman_hip.so is not built")
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("cpu_build") / "filter_staged_cpu"
    cmd = [gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
           "-fno-sanitize-recover=undefined", "-I", str(ROOT / "include"),
           "-I", str(ROOT / "saruman_amd" / "csrc"),
           str(ROOT / "tests" / "cpu_build" / "filter_staged_cpu.cpp"),
           "-L", str(_build.LIBDIR), "-lsaruman_hip", f"-Wl,-rpath,{_build.LIBDIR}", "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("args", [
    ("21", "30000", "600", "36", "36", "60", "0", "0"),
    ("22", "40000", "2000", "40", "40", "7", "1", "0"),
    ("23", "60000", "2000", "36", "250", "50", "1", "1"),
], ids=["uniform", "repeats_tiny_chunks", "mixed_non_acgt"])
def test_staged_lists(exe, args):
    r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("OK"), r.stdout + r.stderr
