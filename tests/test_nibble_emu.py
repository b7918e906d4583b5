"""The band kernels for costs other than 0/1 (saruman_amd/csrc/nw_kernels.hip:
nibble_band_tile and nibble_trace_tile), compiled unmodified for the CPU through a
stand-in HIP header and run lane by lane over random candidates of every band class,
against the oracle (oracle_fill and oracle_traceback, which restate
cuda-functions.cu:413-497 and :108-315): score, transcript and end cell.

Reads of 1-3 bases, of up to 14 (row 0 of every column lies in the band of a candidate
with k >= L, and costs other than its unit steps must not reach the cells below it),
and longer ones on both read-code paths (staged up to 600 codes).  A mistake planted in
the checker must be reported.
"""
import re
import subprocess

import pytest

from test_band_bits_emu import EMU, ROOT, _clang


@pytest.fixture(scope="module")
def emu_bin(tmp_path_factory):
    clang = _clang()
    if clang is None:
        pytest.skip("clang++ not found")
    d = tmp_path_factory.mktemp("emu")
    obj = d / "oracle.o"
    subprocess.run(["gcc", "-O2", "-c", str(ROOT / "oracle" / "nw_oracle.c"), "-o", str(obj)], check=True)
    exe = d / "nibble_emu"
    subprocess.run([clang, "-O2", "-std=c++17", "-I", str(EMU), "-I", str(ROOT / "include"), "-I",
                    str(ROOT / "saruman_amd" / "csrc"), str(EMU / "nibble_emu.cpp"), str(obj), "-o",
                    str(exe)], check=True)
    return exe


def _run(exe, *args):
    r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=300)
    m = re.search(r"cases \d+ hits (\d+) bad (\d+) diag (\d+) top (\d+) left (\d+)", r.stdout)
    assert m, r.stdout + r.stderr
    return r, dict(zip(("hits", "bad", "diag", "top", "left"), map(int, m.groups())))


@pytest.mark.parametrize("match,mismatch", [(0, 1), (0, 2), (0, 3), (1, 3), (5, 2), (5, 1), (40, 7)])
@pytest.mark.parametrize("max_len", [3, 14, 160, 700])
def test_nibble_kernels_match_oracle(emu_bin, match, mismatch, max_len):
    r, t = _run(emu_bin, 4000, 7, match, mismatch, max_len)
    assert r.returncode == 0 and t["bad"] == 0, (t, r.stderr)
    assert t["hits"] > 5 and t["top"] > 50, t


def test_planted_mistake_is_reported(emu_bin):
    r, t = _run(emu_bin, 2000, 3, 0, 2, 14, "plant")
    assert r.returncode == 1 and t["bad"] > 0, t
