"""Buffers that outlive a call are bounded: records of long draws come in
blocks, an ensemble's records go up 64 MiB at a time, a point list's large
workspace is given back.

Tolerance of the draw, before any run: FP64 sums of 1.2e6 harmonics at phases
below 1e4 rad, 1e-10 sigma."""
from __future__ import annotations

import numpy as np
import pytest

from native_lib import build_check, run_check
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


def test_an_ensemble_of_more_records_than_are_staged_at_a_time(lib_f):
    """90 members of 20000 harmonics, 72 MB of records: the members around the
    64 MiB mark and the last are their single runs bit for bit."""
    hip = Hip()
    n = (24, 22, 20)
    members = [dict(nd=3, fe=n, ds=25.0, acf=1, cl=(60.0, 50.0, 40.0), sigma=0.05, hurst=0.3, nharm=20000, seed=q + 1)
               for q in range(90)]
    bufs = [hip.empty(int(np.prod(n)), np.float32) for _ in members]
    print("[case] 90 members of 20000 harmonics", flush=True)
    stats = lib_f.ensemble_execute(members, [b.ptr for b in bufs])
    for q in (0, 82, 83, 84, 89):
        m = members[q]
        init_product(lib_f, structured_cfg(n=n, ds=m["ds"], acf=1, cl=m["cl"], sigma=0.05, hurst=0.3, nharm=20000,
                                           real=np.float32))
        lib_f.set_kernel("auto")
        single, one = lib_f.execute(m["seed"])
        lib_f.finalize()
        assert np.array_equal(bufs[q].numpy(), single.reshape(-1, order="F")), q
        assert np.array_equal(stats[q, :4], one[:4]), q


def test_a_lists_large_workspace_is_given_back(tmp_path):
    out = run_check(build_check("give_back", tmp_path))
    print(out, flush=True)
    assert out.rstrip().endswith("0 bad")
