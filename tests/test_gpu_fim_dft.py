"""FIM grids whose transform runs as dense products on the matrix cores, against the FP64 FIM oracle,
at the edges of that transform's tiles.

A line of length N (even) has N/4 + 1 inputs and outputs per matrix, in steps of 4 and tiles of 16
rows; a block takes 16 columns, or 32 (double: 16) lines along x. An internal length is the grid's
plus one, made even.

Bars as for every FIM grid (test_gpu_fim.py): the products sum at most 256 terms in FP32, whose
rounding (sqrt(256) / 2 units of 6e-8 per axis, 1.5e-6 over three axes) is below the float
library's 1e-5 of the standard deviation, and in FP64 far below 1e-10.
"""
from __future__ import annotations

import numpy as np
import pytest
from test_gpu_fim import _check, _fim, _run, _say

from scarf3d_amd.workloads import structured_cfg

pytestmark = pytest.mark.gpu

# grid (internal lengths): what is at its edge
FLOAT = [
    ((1, 3, 37), "lengths 2, 4 and 38"),
    ((57, 59, 61), "58, 60, 62: up to 16 rows, one tile exactly"),
    ((63, 65, 5), "64, 66: one row in a second tile; 66 x 6 lines, a block of 12"),
    ((121, 45, 11), "122: 31 inputs, a last step of 3; 62 columns, a tile of 14"),
    ((93, 31, 30), "lengths 94 = 2 x 47 and 32, FFT lengths among them"),
    ((617, 20, 4), "618: more than 64 KB of LDS, ten tiles in two turns"),
    ((13, 1017, 6), "1018: 255 rows, 16 tiles in one block"),
    ((1018, 9, 3), "1020 along x: the longest line"),
    ((9, 3, 1009), "1010 along z"),
    ((201, 157, 1), "2D: 202 x 158"),
]
DOUBLE = [FLOAT[0], FLOAT[1], FLOAT[2], FLOAT[3], FLOAT[9],
          ((13, 597, 6), "598: 150 inputs, 152 KB of LDS"),
          ((601, 21, 5), "602 along x")]


def _grid(n, real):
    cl = (900.0, 700.0, 500.0 if n[2] > 1 else 0.0)
    return _fim(structured_cfg(n=n, ds=50.0, cl=cl, hurst=0.3, sigma=0.05, real=real))


@pytest.mark.parametrize("n,why", FLOAT, ids=["x".join(map(str, c[0])) for c in FLOAT])
def test_dense_transform_float(lib_f, n, why):
    _say(n, why)
    _check(lib_f, _grid(n, np.float32), 411, "f")


@pytest.mark.parametrize("n,why", DOUBLE, ids=["x".join(map(str, c[0])) for c in DOUBLE])
def test_dense_transform_double(lib_d, n, why):
    _say(n, why)
    _check(lib_d, _grid(n, np.float64), 412, "d")


def test_tables_follow_the_grid(lib_f, lib_d):
    """Calls that change the grid, the library's type and the transform in turn."""
    for n, lib, flav in (((45, 33, 21), lib_f, "f"), ((45, 21, 33), lib_f, "f"), ((255, 31, 1), lib_f, "f"),
                         ((45, 33, 21), lib_d, "d"), ((45, 33, 21), lib_f, "f")):
        _say(n, flav)
        _check(lib, _grid(n, np.float32 if flav == "f" else np.float64), 413, flav)
        lib.finalize()


# From 2^25 internal points on the transform's last pass writes a block itself. A point of interest
# that reaches no point keeps the field by way of the internal grid: equal bit for bit.
MODEL = (801, 213, 205)  # internal 802 x 214 x 206
BLOCKS = [
    (dict(n=MODEL, ds=25.0), "the whole model"),
    (dict(n=(400, 106, 102), ds=50.0), "nodes without an output"),
    (dict(n=(81, 63, 49), ds=20.0), "nodes with two outputs"),
    (dict(n=(20, 16, 29), fs=(11, 5, 1), ds=25.0), "an inner block"),
    (dict(n=(1, 1, 1), fs=MODEL, ds=25.0), "the model's last point"),
]


@pytest.mark.parametrize("flav", ["f", "d"])
@pytest.mark.parametrize("kw,why", BLOCKS, ids=[b[1].replace(" ", "_") for b in BLOCKS])
def test_blocks_of_the_last_pass(lib_f, lib_d, kw, why, flav):
    lib = lib_f if flav == "f" else lib_d
    got = []
    for poi in (None, np.full((3, 1), -1e6)):
        extra = {} if poi is None else dict(poi=poi, mute=1.0, taper=1.0)
        cfg = structured_cfg(cl=(400.0, 300.0, 200.0), hurst=0.3, sigma=0.05, dh=25.0,
                             real=np.float32 if flav == "f" else np.float64, **kw, **extra)
        cfg["nc"] = (0.0, 0.0, 0.0)
        cfg["fc"] = tuple((n - 1) * 25.0 for n in MODEL)
        _say(why, flav, "through the internal grid" if extra else "")
        field, stats = _run(lib, _fim(cfg), 414)
        lib.finalize()
        got.append((np.array(field), np.array(stats[:4])))
    assert np.any(got[0][0])
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])
