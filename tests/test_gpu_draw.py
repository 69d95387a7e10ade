"""The draw with its trials screened on the GPU against the oracle's draw of
one pair at a time: the FP64 field of the resident record (scarf_srm_run_fp64)
equals the oracle's FP64 field on a small grid to rounding. One harmonic more,
less or elsewhere in the stream moves it by ~1/sqrt(nharm) of sigma.

Tolerance: FP64 sums of <= 12000 harmonics at phases below 1e4 rad, 1e-10 sigma.
"""
from __future__ import annotations

import numpy as np
import pytest

from srm_cases import init_product, oracle_field, structured_cfg

pytestmark = pytest.mark.gpu

# more pairs than the screen's threshold in every case
CASES = [
    ("vk", dict(n=(9, 8, 7), cl=(300.0, 200.0, 250.0), hurst=0.25, nharm=6000), 0),
    ("vk_rare", dict(n=(60, 50, 2), cl=(250.0, 200.0, 300.0), hurst=0.5, dh=2.0, nharm=3000, box=1000.0), 0),
    # the spectrum's maximum inside the band: bins without a bound
    ("gauss", dict(n=(12, 11, 10), acf=1, cl=(300.0, 300.0, 300.0), nharm=12000, box=6000.0), 0),
    ("vk_max_in_band", dict(n=(12, 11, 10), cl=(100.0, 90.0, 80.0), hurst=0.9, nharm=5000, box=3000.0), 0),
    ("2d", dict(n=(30, 20, 1), cl=(150.0, 120.0, 0.0), hurst=0.3, nharm=5000), 0),
    # harmonics dropped above kc: two pairs consumed instead of four
    ("dropped", dict(n=(20, 18, 16), cl=(200.0, 150.0, 180.0), hurst=0.1, dh=10.0, nharm=4000), 0),
    # blocks that end between a trial and its pairs
    ("small_blocks", dict(n=(9, 8, 7), cl=(300.0, 200.0, 250.0), hurst=0.25, nharm=1500), 37),
    ("blocks", dict(n=(9, 8, 7), cl=(300.0, 200.0, 250.0), hurst=0.25, nharm=6000), 2049),
]


@pytest.mark.parametrize("name,kw,block", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("flavour", ["f", "d"])
def test_screened_draw_is_the_oracles(request, oracle, flavour, name, kw, block):
    from scarf3d_amd.hip import Hip

    lib = request.getfixturevalue("lib_" + flavour)
    kw = dict(kw)
    box = kw.pop("box", None)
    cfg = structured_cfg(ds=50.0, real=lib.dtype, **kw)
    if box:
        cfg["fc"] = (box, box, box if cfg["nd"] == 3 else 0.0)
    hip = Hip()
    for seed in (1234, 77, 2_000_000_011):
        print("[case]", flavour, name, seed, flush=True)
        ref, s = oracle_field(oracle, cfg, seed, flavour)
        init_product(lib, cfg)
        if block:
            assert lib.set_option("draw_block", block) == 0
        n, _ = lib.srm_draw(seed)
        d = hip.empty(int(np.prod(cfg["fe"])), np.float64)
        lib.srm_run_fp64(d.ptr)
        lib.set_option("draw_block", 0)
        lib.finalize()
        err = np.abs(d.numpy() - np.asarray(ref).reshape(-1, order="F")).max() / cfg["sigma"]
        print(f"  kept {n} of {cfg['nharm']}, max {err:.2e} sigma", flush=True)
        assert err <= 1e-10


# a wave's share of the stream: one round of 64 pairs, a few, all 32; one group
# of chunks put in order, with a remainder, and many
SIZES = [dict(nharm=130, dh=50.0), dict(nharm=1501, dh=20.0), dict(nharm=9001, dh=4.0), dict(nharm=12000, dh=2.0)]


@pytest.mark.parametrize("kw", SIZES, ids=[str(k["nharm"]) for k in SIZES])
@pytest.mark.parametrize("flavour", ["f", "d"])
def test_short_and_long_screened_draws(request, oracle, flavour, kw):
    test_screened_draw_is_the_oracles(request, oracle, flavour, "sizes",
                                      dict(n=(9, 8, 3), cl=(300.0, 200.0, 250.0), hurst=0.4, box=1000.0, **kw), 0)
