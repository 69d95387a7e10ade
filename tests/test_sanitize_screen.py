"""The screened draw (CPU, sanitized): tests/sanitize/screened_draw_check.cpp,
g++ -fsanitize=address,undefined on the product's own host sources, runs
HarmonicSampler::create_rows through a host TrialScreen and compares its rows
bit for bit with the unscreened draw's, which test_host_parity.py holds
against the oracle."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "scarf3d_amd" / "csrc"


def test_screened_rows_equal_the_unscreened_draws(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not found")
    exe = tmp_path / "screened_draw_check"
    flags = ["-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer", "-fsanitize=address,undefined",
             "-fno-sanitize-recover=all", "-ffp-contract=off", "-fno-fast-math", "-fno-builtin-sin",
             "-fno-builtin-cos", "-fno-builtin-sinf", "-fno-builtin-cosf", "-fno-builtin-sincos",
             "-fno-builtin-sincosf", "-pthread", "-I", str(CSRC)]
    srcs = [ROOT / "tests" / "sanitize" / "screened_draw_check.cpp", CSRC / "srm_host.cpp", CSRC / "quadpack.cpp"]
    res = subprocess.run([gxx, *flags, *map(str, srcs), "-o", str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300,
                         env={"ASAN_OPTIONS": "detect_leaks=1:abort_on_error=1", "PATH": "/usr/bin:/bin"})
    assert run.returncode == 0, run.stdout[-3000:] + run.stderr[-3000:]
    assert "runtime error" not in run.stderr and "AddressSanitizer" not in run.stderr, run.stderr[-3000:]
    assert run.stdout.rstrip().endswith("0 bad")
    # pairs left open, rejected ones and several blocks did occur
    counts = [[int(f.split()[0]) for f in line.split(":")[1].split(",")] for line in run.stdout.splitlines() if " held," in line]
    assert max(c[0] for c in counts) > 3 and max(c[2] for c in counts) > 0 and max(c[3] for c in counts) > 0
