"""A thin block of many planes and many harmonics by the fast transform, with a
SCARF_DEVICE_MEMORY_LIMIT that its bounded workspace satisfies (the harmonics'
values of all planes at once would take 4 GB, the direct sum's tables 2 GB),
against the direct FP64 sum.

Tolerance, before any run: the transform's in double (1e-11 of the standard
deviation)."""
from __future__ import annotations

import numpy as np
import pytest

from scarf3d_amd.hip import Hip
from scarf3d_amd.workloads import init_library, structured_cfg

pytestmark = pytest.mark.gpu


def test_a_tall_block_within_a_limit(lib_d, monkeypatch):
    n = (30, 30, 8192)
    cfg = structured_cfg(n=n, ds=20.0, cl=(300.0, 300.0, 900.0), hurst=0.25, nharm=30000, real=np.float64)
    d = Hip().empty(int(np.prod(n)), np.float64)
    init_library(lib_d, cfg)
    lib_d.set_kernel("auto")
    monkeypatch.setenv("SCARF_DEVICE_MEMORY_LIMIT", "1")
    with pytest.raises(RuntimeError) as refused:
        lib_d.srm_draw(3)
    held = int(str(refused.value).split("library holds ")[1].split()[0])  # from earlier tests
    monkeypatch.setenv("SCARF_DEVICE_MEMORY_LIMIT", str(held + (600 << 20)))
    print("[case]", n, "held", held, flush=True)
    lib_d.srm_draw(3)
    lib_d.srm_run(d.ptr)
    out = d.numpy().copy()
    monkeypatch.delenv("SCARF_DEVICE_MEMORY_LIMIT")
    lib_d.set_kernel("direct_f64")
    lib_d.srm_run(d.ptr)
    ref = d.numpy()
    lib_d.set_kernel("auto")
    lib_d.finalize()
    err = np.abs(out - ref).max() / ref.std()
    print(f"  max {err:.2e} sigma", flush=True)
    assert 0 < err <= 1e-11
