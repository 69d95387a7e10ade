"""Point lists under `auto`, interpolated from a grid by the fast transform,
against the direct FP64 sum of the same draw (scarf_srm_run_fp64).

Tolerances, before any run: the transform's (test_gpu_transform.py) plus the
interpolation's kernel error (2e-8, 1e-14) and one more rounding: 1e-5 of the
standard deviation at any point and 8e-7 in the 2-norm in float; 1e-11 in
double (1e-10 for points 1e6 m from the origin, phases of 1e5 rad).
"""
from __future__ import annotations

import numpy as np
import pytest

from scarf3d_amd.hip import Hip
from scarf3d_amd.workloads import init_library, unstructured_cfg

pytestmark = pytest.mark.gpu

BOX = dict(box=(3000.0, 2500.0, 2000.0), dh=50.0, acf=0, hurst=0.25, cl=(400.0, 300.0, 300.0), nharm=4000)


def _run(lib, cfg, seed=6):
    """(auto's field and statistics, FP64 field, the direct kernel's field)"""
    hip = Hip()
    init_library(lib, cfg)
    lib.set_kernel("auto")
    lib.srm_draw(seed)
    n = len(cfg["x"])
    d, d64 = hip.empty(n, lib.dtype), hip.empty(n, np.float64)
    st = lib.srm_run(d.ptr)
    out = d.numpy().copy()
    lib.srm_run(d.ptr)
    assert np.array_equal(d.numpy(), out, equal_nan=True)
    lib.srm_run_fp64(d64.ptr)
    lib.set_kernel("direct_f32" if lib.flavour == "f" else "direct_f64")
    lib.srm_run(d.ptr)
    direct = d.numpy().copy()
    lib.set_kernel("auto")
    lib.finalize()
    return out, st, d64.numpy(), direct


def _cfg(lib, npts, box=None, **kw):
    c = unstructured_cfg(npts=npts, real=lib.dtype, **{**BOX, **({"box": box} if box else {}), **kw})
    for a in "xyz":
        c[a] = c[a].astype(lib.dtype)
    return c


def _check(lib, cfg, bar_d=1e-11, same_ok=False):
    out, st, ref, direct = _run(lib, cfg)
    sd = max(ref.std(), 0.3 * cfg["sigma"])
    err = np.abs(out - ref).max() / sd
    rms = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"  max {err:.2e} sigma, 2-norm {rms:.2e}", flush=True)
    assert same_ok or not np.array_equal(out, direct)
    assert err <= (1e-5 if lib.flavour == "f" else bar_d)
    if len(out) > 100:
        assert rms <= (8e-7 if lib.flavour == "f" else bar_d)
    if len(out) > 100 and not cfg["rescale"]:  # a rescale reports sigma and 0
        v = out.astype(np.float64)
        assert abs(float(st[2]) / v.std(ddof=1) - 1) <= (2e-7 if lib.flavour == "f" else 1e-12)
        assert abs(float(st[3]) - v.mean()) <= (2e-7 if lib.flavour == "f" else 1e-12) * sd


@pytest.mark.parametrize("flavour", ["f", "d"])
@pytest.mark.parametrize("npts", [1, 2, 7, 33, 4095, 4097, 30011, 250000])
def test_counts(request, flavour, npts):
    lib = request.getfixturevalue("lib_" + flavour)
    cfg = _cfg(lib, npts)
    cfg["nc"], cfg["fc"] = (0.0, 0.0, 0.0), (3000.0, 2500.0, 2000.0)
    print("[case]", flavour, npts, flush=True)
    if npts == 1:
        out, _, ref, _ = _run(lib, cfg)
        assert np.abs(out - ref).max() <= (1e-5 if flavour == "f" else 1e-11) * cfg["sigma"]
    else:
        _check(lib, cfg, same_ok=npts < 4)


CASES = [
    ("gaussian", dict(acf=1, cl=(800.0, 700.0, 500.0), nharm=8000), None),
    ("2d", dict(nd=2, cl=(300.0, 400.0, 0.0), nharm=5000), None),
    ("flat_box", dict(box=(9000.0, 8000.0, 120.0)), "model"),
    ("one_line", dict(), "line"),
    ("clustered", dict(), "cluster"),
    ("far", dict(), "far"),
    ("rotated", dict(alpha=25.0, beta=-40.0, gamma=10.0), None),
    ("rescale_taper", dict(rescale=1, poi=np.array([[500.0, 2000.0], [900.0, 1500.0], [400.0, 300.0]]), mute=100.0,
                           taper=500.0), None),
]


@pytest.mark.parametrize("flavour", ["f", "d"])
@pytest.mark.parametrize("name,kw,how", CASES, ids=[c[0] for c in CASES])
def test_lists_match_the_direct_sum(request, flavour, name, kw, how):
    lib = request.getfixturevalue("lib_" + flavour)
    cfg = _cfg(lib, 20000, **kw)
    if how == "line":
        cfg["y"][:] = 777.0
    elif how == "cluster":
        for a in "xyz":
            cfg[a][:19990] = (cfg[a][:19990] * lib.dtype(1e-3) + lib.dtype(400.0)).astype(lib.dtype)
    elif how == "far":
        for a in "xyz":
            cfg[a] += lib.dtype(1.0e6)
    if how:
        cfg["nc"] = (0.0, 0.0, 0.0)
        cfg["fc"] = (9000.0, 8000.0, 4000.0)
        if how == "far":
            cfg["nc"], cfg["fc"] = (1.0e6,) * 3, (1.003e6, 1.0025e6, 1.002e6)
    print("[case]", flavour, name, flush=True)
    if name == "rescale_taper":
        cfg["poi"] = cfg["poi"].astype(lib.dtype)
    _check(lib, cfg, 1e-10 if how == "far" else 1e-11)


def test_not_a_number_stays_at_its_point(lib_f):
    cfg = _cfg(lib_f, 5000)
    cfg["x"][17] = np.nan
    cfg["z"][4000] = np.nan
    cfg["nc"], cfg["fc"] = (0.0, 0.0, 0.0), (3000.0, 2500.0, 2000.0)
    out, _, ref, _ = _run(lib_f, cfg)
    assert np.array_equal(np.isnan(out), np.isnan(ref)) and np.isnan(out).sum() == 2
    ok = ~np.isnan(ref)
    assert np.abs(out[ok] - ref[ok]).max() <= 1e-5 * ref[ok].std()


def test_an_infinite_coordinate_takes_the_direct_sum(lib_f):
    cfg = _cfg(lib_f, 5000)
    cfg["y"][3] = np.inf
    cfg["nc"], cfg["fc"] = (0.0, 0.0, 0.0), (3000.0, 2500.0, 2000.0)
    out, _, _, direct = _run(lib_f, cfg)
    assert np.array_equal(out, direct, equal_nan=True)
