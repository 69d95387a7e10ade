"""The fast transform that `auto` takes on grids of more than a few hundred
harmonics, against the direct FP64 sum of the same draw (scarf_srm_run_fp64,
which test_gpu_parity.py holds against the oracle) and the direct kernels.

Tolerances, before any run. Float: the Kaiser-Bessel kernel's error (2e-8 of
the field's rms at 9 taps and oversampling 1.9) and FP32 rounding of two
transforms of up to 2^13 values, about 0.5 eps per level and axis with eps =
6e-8: 8e-7 in the 2-norm; 1e-5 of the standard deviation at any point, the bar
of every float kernel. Double: 16 taps, 1e-14 kernel error, phases of up to
1e4 rad at eps = 1.1e-16: 1e-11 at any point.
"""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from scarf3d_amd.hip import Hip
from scarf3d_amd.workloads import init_library, structured_cfg

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parents[1]


def _fields(lib, cfg, seed, kernel="auto"):
    """(field of `kernel`, its statistics, FP64 field, direct_f32 field)."""
    hip = Hip()
    init_library(lib, cfg)
    assert lib.set_kernel(kernel) == 0
    n = int(np.prod([cfg["fe"][i] - cfg["fs"][i] + 1 for i in range(3)]))
    lib.srm_draw(seed)
    d, d64 = hip.empty(n, lib.dtype), hip.empty(n, np.float64)
    stats = lib.srm_run(d.ptr)
    out = d.numpy().copy()
    lib.srm_run_fp64(d64.ptr)
    lib.set_kernel("direct_f32")
    lib.srm_run(d.ptr)
    direct = d.numpy().copy()
    lib.set_kernel("auto")
    lib.finalize()
    return out, stats, d64.numpy(), direct


def _check(lib, cfg, seed):
    out, stats, ref, direct = _fields(lib, cfg, seed)
    assert not np.array_equal(out, direct)  # the transform ran, not the direct kernel
    sd = ref.std()
    err = np.abs(out.astype(np.float64) - ref).max() / sd
    rms = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"  max {err:.2e} sigma, 2-norm {rms:.2e}", flush=True)
    bar, bar2 = (1e-5, 8e-7) if lib.flavour == "f" else (1e-11, 1e-11)
    assert err <= bar and rms <= bar2
    if not cfg["rescale"]:
        v = out.astype(np.float64)
        assert abs(float(stats[2]) / v.std(ddof=1) - 1) <= (2e-7 if lib.flavour == "f" else 1e-12)
        assert abs(float(stats[3]) - v.mean()) <= (2e-7 if lib.flavour == "f" else 1e-12) * sd
    return out


# every transform length m * 2^a of either axis: n just below length / 1.9
LENGTHS = {m: [m << a for a in range(5, 14) if m << a <= 8192] for m in (1, 3, 5, 7, 9)}


@pytest.mark.parametrize("m", sorted(LENGTHS))
@pytest.mark.parametrize("flavour", ["f", "d"])
def test_every_transform_length(request, m, flavour):
    lib = request.getfixturevalue("lib_" + flavour)
    most = 8192 if flavour == "f" else 4096
    sizes = [int(v / 1.9) for v in LENGTHS[m] if v <= most]
    for a, b in zip(sizes, reversed(sizes)):
        cfg = structured_cfg(n=(a, b, 1), ds=10.0, cl=(max(25.0, 0.1 * 10 * min(a, b)),) * 2 + (0.0,), hurst=0.3,
                             nharm=1200, real=lib.dtype)
        print("[case]", flavour, (a, b), flush=True)
        _check(lib, cfg, 11)


SHAPES = [
    ("cube", dict(n=(33, 32, 31), cl=(200.0, 150.0, 120.0))),
    # thin blocks of a model of 100 points per axis
    ("thin_x", dict(n=(1, 70, 90), cl=(200.0, 200.0, 200.0))),
    ("thin_y", dict(n=(90, 2, 70), cl=(200.0, 200.0, 200.0))),
    ("thin_z", dict(n=(100, 97, 1), cl=(300.0, 300.0, 200.0))),
    ("ragged_z", dict(n=(40, 150, 201), cl=(100.0, 300.0, 300.0))),
    ("rotated", dict(n=(65, 47, 29), cl=(200.0, 150.0, 120.0), alpha=35.0, beta=-20.0, gamma=50.0)),
    ("gaussian", dict(n=(96, 80, 64), acf=1, cl=(250.0, 200.0, 150.0))),
    ("finer_ds", dict(n=(64, 64, 48), dh=25.0, cl=(200.0, 200.0, 150.0))),
    ("coarser_ds", dict(n=(64, 64, 48), dh=5.0, cl=(200.0, 200.0, 150.0))),
    ("rescale_taper", dict(n=(64, 48, 40), cl=(200.0, 150.0, 120.0), rescale=1,
                           poi=np.array([[100.0, 400.0], [200.0, 150.0], [50.0, 300.0]]), mute=40.0, taper=100.0)),
]


@pytest.mark.parametrize("name,kw", SHAPES, ids=[s[0] for s in SHAPES])
@pytest.mark.parametrize("flavour", ["f", "d"])
def test_shapes_match_the_direct_sum(request, flavour, name, kw):
    lib = request.getfixturevalue("lib_" + flavour)
    cfg = structured_cfg(ds=10.0, nharm=3001, real=lib.dtype, **{"hurst": 0.25, **kw})
    if name.startswith("thin"):
        cfg["fc"] = (990.0,) * 3
    _check(lib, cfg, 5)


def test_most_harmonics_in_few_classes(lib_f):
    """A Gaussian spectrum on a box of few correlation lengths: nearly every
    harmonic falls on the same few frequencies (the classes all waves share)."""
    cfg = structured_cfg(n=(200, 180, 30), ds=10.0, acf=1, cl=(680.0, 600.0, 95.0), nharm=20000, real=np.float32)
    _check(lib_f, cfg, 3)


def test_slabs_equal_the_whole_and_repeat(lib_f):
    """Planes are independent: z slabs of a larger model, by fs/fe and nc/fc,
    are the whole field's planes bit for bit; and a run repeats."""
    kw = dict(ds=20.0, cl=(500.0, 400.0, 300.0), hurst=0.2, nharm=4000, real=np.float32)
    whole = structured_cfg(n=(120, 100, 60), **kw)
    a = _check(lib_f, whole, 9).reshape((120, 100, 60), order="F")
    assert np.array_equal(a, _fields(lib_f, whole, 9)[0].reshape(a.shape, order="F"))
    for z0, nz in ((0, 17), (17, 1), (18, 42)):
        cfg = structured_cfg(n=(120, 100, nz), fs=(1, 1, z0 + 1), **kw)
        cfg["nc"], cfg["fc"] = whole["nc"], whole["fc"]
        b = _fields(lib_f, cfg, 9)[0].reshape((120, 100, nz), order="F")
        assert np.array_equal(b, a[:, :, z0:z0 + nz]), z0


def test_block_offsets_along_x_and_y(lib_d):
    kw = dict(ds=20.0, cl=(500.0, 400.0, 300.0), hurst=0.2, nharm=2000, alpha=20.0, real=np.float64)
    whole = structured_cfg(n=(90, 80, 20), **kw)
    a = _check(lib_d, whole, 9).reshape((90, 80, 20), order="F")
    cfg = structured_cfg(n=(50, 37, 20), fs=(31, 12, 1), **kw)
    cfg["nc"], cfg["fc"] = whole["nc"], whole["fc"]
    b = _check(lib_d, cfg, 9).reshape((50, 37, 20), order="F")
    assert np.abs(b - a[30:80, 11:48]).max() <= 1e-11 * a.std()


def test_without_room_the_direct_kernel_runs():
    """SCARF_DEVICE_MEMORY_LIMIT below the transform's workspace but above the
    direct kernel's tables: auto gives the direct kernel's field."""
    code = """
import numpy as np, os, scarf3d_amd
from scarf3d_amd.workloads import structured_cfg, init_library
lib = scarf3d_amd.load("f")
cfg = structured_cfg(n=(150, 130, 100), ds=20.0, cl=(500.0, 400.0, 300.0), hurst=0.2, nharm=500)
def field(kernel, limit):
    os.environ.pop("SCARF_DEVICE_MEMORY_LIMIT", None)
    if limit: os.environ["SCARF_DEVICE_MEMORY_LIMIT"] = str(limit)
    init_library(lib, cfg); lib.set_kernel(kernel)
    f, st = lib.execute(4); e = lib.last_error(); lib.finalize()
    assert e == "", e
    return f.copy()
tight = field("auto", 12 << 20)
direct = field(DIRECT, 0)
free = field("auto", 0)
assert np.array_equal(tight, direct) and not np.array_equal(free, direct)
assert np.abs(free - direct).max() <= 1e-5 * direct.std()
print("ok")
"""
    # 382 column tiles of 256 x 2 x tiles: the kernel auto names for this grid
    import scarf3d_amd

    lib = scarf3d_amd.load("f")
    init_library(lib, structured_cfg(n=(150, 130, 100), ds=20.0, cl=(500.0, 400.0, 300.0), hurst=0.2, nharm=500))
    lib.set_kernel("auto")
    direct = lib.kernel()
    lib.finalize()
    r = subprocess.run([sys.executable, "-c", code.replace("DIRECT", repr(direct))], cwd=ROOT, capture_output=True,
                       text=True, timeout=100, env={**os.environ, "SCARF_TUNE": "0"})
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


def _members(nharm, n=6):
    out = []
    for q in range(n):
        out.append(dict(fe=(60 + 17 * q, 50 + 9 * q, 24 + 5 * q), ds=25.0, acf=q % 2, cl=(300.0, 250.0, 180.0), sigma=0.05,
                        hurst=0.1 + 0.1 * q, nharm=nharm + 64 * q, seed=q + 1, rescale=int(q == 2),
                        alpha=10.0 * (q == 3)))
    out[4].update(nd=2, fe=(210, 150, 1), cl=(400.0, 300.0, 0.0))
    return out


@pytest.mark.parametrize("flavour", ["f", "d"])
def test_ensemble_members_equal_single_runs(request, flavour):
    """Under auto an ensemble of many harmonics runs its members by the
    transform: each is its single run bit for bit, and a table drawn before
    stays resident."""
    lib = request.getfixturevalue("lib_" + flavour)
    hip = Hip()
    members = _members(3000)
    bufs = [hip.empty(int(np.prod(m["fe"])), lib.dtype) for m in members]
    cfg = structured_cfg(n=(40, 30, 20), ds=25.0, cl=(300.0, 250.0, 180.0), nharm=2000, real=lib.dtype)
    init_library(lib, cfg)
    lib.set_kernel("auto")
    lib.srm_draw(5)
    d = hip.empty(40 * 30 * 20, lib.dtype)
    lib.srm_run(d.ptr)
    before = d.numpy().copy()
    for _ in range(2):
        stats = lib.ensemble_execute(members, [b.ptr for b in bufs])
    lib.srm_run(d.ptr)
    assert np.array_equal(d.numpy(), before)
    lib.finalize()
    for m, b, st in zip(members, bufs, stats):
        print("[case]", flavour, m["fe"], m["nharm"], flush=True)
        c = structured_cfg(n=m["fe"], ds=m["ds"], acf=m["acf"], cl=m["cl"], sigma=m["sigma"], hurst=m["hurst"],
                           nharm=m["nharm"], alpha=m["alpha"], rescale=m["rescale"], real=lib.dtype)
        init_library(lib, c)
        single, one = lib.execute(m["seed"])
        lib.finalize()
        assert np.array_equal(b.numpy(), single.reshape(-1, order="F"))
        assert np.array_equal(st[:4], one[:4])


def test_ensemble_of_few_harmonics_is_grouped(lib_f):
    hip = Hip()
    members = [dict(m, nd=3, fe=(600, 500, 40), cl=(600.0, 500.0, 200.0)) for m in _members(64)]
    bufs = [hip.empty(int(np.prod(m["fe"])), np.float32) for m in members]
    a = lib_f.ensemble_execute(members, [b.ptr for b in bufs])
    fields = [b.numpy().copy() for b in bufs]
    b_ = lib_f.ensemble_execute(members, [b.ptr for b in bufs], "mfma_bf16x3")
    assert np.array_equal(a[:, :4], b_[:, :4])
    assert all(np.array_equal(f, b.numpy()) for f, b in zip(fields, bufs))


WIDE = [(dict(n=(60, 1000, 13), cl=(120.0, 900.0, 40.0)), "fd"), (dict(n=(35, 2100, 9), cl=(100.0, 1500.0, 30.0)), "f"),
        (dict(n=(41, 500, 9), cl=(100.0, 500.0, 30.0)), "d"), (dict(n=(33, 1100, 5), cl=(100.0, 900.0, 20.0)), "d"),
        (dict(n=(60, 1000, 13), cl=(190.0, 3000.0, 40.0), acf=1, nharm=20000), "f"),
        (dict(n=(60, 500, 13), cl=(190.0, 1500.0, 40.0), acf=1, nharm=20000), "d")]


@pytest.mark.parametrize("kw,flavour", [(kw, f) for kw, fs in WIDE for f in fs])
def test_long_lines_with_the_unit_to_themselves(request, kw, flavour):
    """Lines of which eight planes fill more than half of a compute unit's LDS:
    one block of 1024 threads each; also with most harmonics in few classes."""
    lib = request.getfixturevalue("lib_" + flavour)
    _check(lib, structured_cfg(ds=10.0, real=lib.dtype, **{"hurst": 0.25, "nharm": 3001, **kw}), 7)


@pytest.mark.parametrize("nx", [64, 66, 67])
@pytest.mark.parametrize("flavour", ["f", "d"])
def test_fields_at_any_alignment(request, flavour, nx):
    """Values are stored in pairs where rows and field allow it: the same bits
    one value off, where they do not."""
    lib = request.getfixturevalue("lib_" + flavour)
    hip = Hip()
    init_library(lib, structured_cfg(n=(nx, 50, 20), ds=10.0, cl=(100.0, 90.0, 50.0), hurst=0.25, nharm=2000,
                                     real=lib.dtype))
    lib.set_kernel("auto")
    lib.srm_draw(3)
    n = nx * 50 * 20
    d = hip.empty(n + 1, lib.dtype)
    a = lib.srm_run(d.ptr)
    at = d.numpy()[:n].copy()
    b = lib.srm_run(d.ptr + np.dtype(lib.dtype).itemsize)
    assert np.array_equal(at, d.numpy()[1:]) and np.array_equal(a[:4], b[:4])
    lib.finalize()
