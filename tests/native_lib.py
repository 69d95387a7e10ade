"""Checks written in C++ against the library's internal headers: compiled for
the host alone and linked with the built library."""
from __future__ import annotations

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
HIPCC = "/opt/rocm/bin/hipcc"


def build_check(name: str, out_dir, flavour: str = "f") -> Path:
    """tests/native/<name>.cpp as a program of library `flavour`."""
    lib = ROOT / "scarf3d_amd" / "lib"
    exe = Path(out_dir) / f"{name}_{flavour}"
    cmd = [HIPCC, "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-O1", "-Wall",
           "-Wno-unused-function", "-I", str(ROOT / "scarf3d_amd" / "csrc"), "-I", str(ROOT / "include"),
           str(ROOT / "tests" / "native" / f"{name}.cpp"), "-o", str(exe), "-L", str(lib),
           "-lscarf3df" if flavour == "f" else "-lscarf3d", "-ldl", f"-Wl,-rpath,{lib}"]
    if flavour == "d":
        cmd.insert(6, "-DDOUBLE_PREC")
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return exe


def run_check(exe: Path, *args, timeout: int = 100, env=None) -> str:
    res = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=timeout, env=env)
    assert res.returncode == 0, f"status {res.returncode}\n{res.stdout[-3000:]}{res.stderr[-3000:]}"
    return res.stdout
