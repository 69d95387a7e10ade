"""Buffers that outlive a call are bounded: records of long draws come in
blocks.

Tolerance of the draw, before any run: FP64 sums of 1.2e6 harmonics at phases
below 1e4 rad, 1e-10 sigma."""
from __future__ import annotations

import numpy as np
import pytest

from scarf3d_amd.hip import Hip
from srm_cases import init_product, oracle_field, structured_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flavour", ["f", "d"])
def test_a_draw_of_several_blocks_of_records(request, oracle, flavour):
    """More than 2^20 records: each harmonic is one at least."""
    lib = request.getfixturevalue("lib_" + flavour)
    cfg = structured_cfg(n=(5, 4, 3), ds=50.0, cl=(300.0, 300.0, 300.0), acf=1, nharm=1200000, real=lib.dtype)
    cfg["fc"] = (6000.0,) * 3
    print("[case]", flavour, cfg["nharm"], flush=True)
    ref, _ = oracle_field(oracle, cfg, 77, flavour)
    init_product(lib, cfg)
    n, _ = lib.srm_draw(77)
    d = Hip().empty(60, np.float64)
    lib.srm_run_fp64(d.ptr)
    lib.finalize()
    err = np.abs(d.numpy() - np.asarray(ref).reshape(-1, order="F")).max() / cfg["sigma"]
    print(f"  kept {n}, max {err:.2e} sigma", flush=True)
    assert n > 1 << 20 and err <= 1e-10
