"""The device filter's batch pass (saruman_amd/csrc/filter_batch.h), compiled for the
host under ASan and UBSan, against the host's pass over random entries: flushes of a
few reads, genome ends and separators, and entries skipped there (whose reads later
flushes walk again)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    from saruman_amd import _build
    gxx = shutil.which("g++")
    if gxx is None or not _build.LIB.exists():
        pytest.skip("g++ or libsaruman_hip.so not available")
    out = tmp_path_factory.mktemp("cpu_build") / "filter_batch_cpu"
    cmd = [gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
           "-fno-sanitize-recover=undefined", "-I", str(ROOT / "include"),
           "-I", str(ROOT / "saruman_amd" / "csrc"),
           str(ROOT / "tests" / "cpu_build" / "filter_batch_cpu.cpp"),
           "-L", str(_build.LIBDIR), "-lsaruman_hip", f"-Wl,-rpath,{_build.LIBDIR}", "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_batch_pass_parts(exe, seed):
    r = subprocess.run([str(exe), str(seed), "4000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("OK"), r.stdout + r.stderr
    assert "left_out=0 " not in r.stdout    # the walk had work


def test_planted_mistake_is_reported(exe):
    r = subprocess.run([str(exe), "4", "500", "plant"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 1 and r.stdout.startswith("MISMATCH"), r.stdout + r.stderr
