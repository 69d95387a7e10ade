"""A point list interpolated in more than one launch (2^18 blocks of 32 points
each in float, of 16 in double), with the last one's ragged end, against the
direct FP64 sum.

Tolerances, before any run: those of the interpolated lists (1e-5 of the
standard deviation at any point in float, 1e-11 in double).
"""
from __future__ import annotations

import numpy as np
import pytest

from scarf3d_amd.hip import Hip
from scarf3d_amd.workloads import init_library, unstructured_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flavour,npts,bar", [("f", (1 << 23) + 77, 1e-5), ("d", (1 << 22) + 33, 1e-11)])
def test_lists_of_two_launches(request, flavour, npts, bar):
    lib = request.getfixturevalue("lib_" + flavour)
    hip = Hip()
    cfg = unstructured_cfg(npts=npts, box=(3000.0, 2500.0, 2000.0), dh=50.0, acf=0, hurst=0.25,
                           cl=(400.0, 300.0, 300.0), nharm=4000, real=lib.dtype)
    print("[case]", flavour, npts, flush=True)
    init_library(lib, cfg)
    lib.set_kernel("auto")
    lib.srm_draw(6)
    d, d64 = hip.empty(npts, lib.dtype), hip.empty(npts, np.float64)
    lib.srm_run(d.ptr)
    out = d.numpy().copy()
    lib.srm_run_fp64(d64.ptr)
    ref = d64.numpy()
    lib.set_kernel("direct_f32" if flavour == "f" else "direct_f64")
    lib.srm_run(d.ptr)
    assert not np.array_equal(d.numpy(), out)  # interpolated, not summed
    lib.set_kernel("auto")
    lib.finalize()
    err = np.abs(out - ref) / ref.std()
    print(f"  max {err.max():.2e} sigma, in the last launch {err[npts // 2:].max():.2e}", flush=True)
    assert err.max() <= bar
