"""The grid epilogue's line-by-line choice of the points of interest against a
statement of the taper at every point: the field with points of interest equals
the field without, times each one's factor in order, at `real` precision.

Tolerance: the factor's operations are the library's own in its precision
(IEEE sums, products and square root); its cosine is the GPU's, a few ulp from
numpy's, on a factor of at most 1 per point of interest: 1e-6 (1e-14) of the
field's largest value.
"""
from __future__ import annotations

import numpy as np
import pytest

from scarf3d_amd.workloads import init_library, structured_cfg

pytestmark = pytest.mark.gpu

CASES = [
    ("line_of_one", dict(n=(1, 30, 20)), 3, 20.0, 90.0),
    ("ragged", dict(n=(67, 31, 9)), 5, 20.0, 90.0),
    ("long_lines", dict(n=(517, 12, 7)), 2, 30.0, 200.0),
    ("two_groups", dict(n=(130, 24, 10)), 130, 10.0, 25.0),
    ("no_taper", dict(n=(64, 33, 8)), 4, 60.0, 1e-3),
    ("wide", dict(n=(65, 20, 8)), 6, 50.0, 4000.0),
    ("flat", dict(n=(90, 70, 1)), 7, 40.0, 80.0),
    ("offset", dict(n=(50, 40, 12), fs=(9, 5, 3)), 4, 20.0, 90.0),
]


@pytest.mark.parametrize("name,kw,npoi,mute,taper", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("flavour", ["f", "d"])
@pytest.mark.parametrize("rescale", [0, 1])
def test_tapers_by_line(request, flavour, name, kw, npoi, mute, taper, rescale):
    lib = request.getfixturevalue("lib_" + flavour)
    r = lib.dtype
    flat = kw["n"][2] == 1
    base = structured_cfg(ds=10.0, cl=(120.0, 100.0, 0.0 if flat else 90.0), nharm=150, real=r, **kw)
    base["fc"] = tuple(1000.0 if d < base["nd"] else 0.0 for d in range(3))
    base["nc"] = (0.0, 0.0, 0.0)
    base["rescale"] = rescale
    n = kw["n"]
    rng = np.random.default_rng(npoi)
    nd = base["nd"]
    poi = (np.array(base["fs"][:nd])[:, None] - 1 + rng.uniform(-0.2, 1.2, (nd, npoi)) * np.array(n[:nd])[:, None]) * 10.0
    poi = poi.astype(r)

    def field(cfg):
        init_library(lib, cfg)
        lib.set_kernel("direct_f64")
        f, _ = lib.execute(8)
        assert lib.last_error() == ""
        lib.set_kernel("auto")
        lib.finalize()
        return f.reshape(n, order="F").copy()

    plain = field(base)
    got = field(dict(base, poi=poi, mute=float(r(mute)), taper=float(r(taper))))
    want = plain.copy()
    ax = [(np.arange(n[d]) + base["fs"][d] - 1).astype(r) * r(10.0) for d in range(3)]
    for q in range(npoi):
        p = [poi[d, q] if d < nd else r(0) for d in range(3)]
        dx, dy, dz = (ax[0] - p[0])[:, None, None], (ax[1] - p[1])[None, :, None], (ax[2] - p[2])[None, None, :]
        d = np.sqrt((dx * dx + dy * dy) + dz * dz)
        t = (d - r(mute)) / r(taper)
        ramp = (d > r(mute)) & (d <= r(mute) + r(taper))
        f = np.where(ramp, r(0.5) - r(0.5) * np.cos(np.where(ramp, t, r(0)) * r(np.pi)), r(1))
        want = np.where(d <= r(mute), r(0), want * f).astype(r)
    bar = (1e-6 if flavour == "f" else 1e-14) * np.abs(plain).max()
    assert np.abs(got - want).max() <= bar
    assert np.array_equal(got == 0, want == 0)
    assert name == "wide" or np.any(got == plain) or npoi > 64
