"""Ensembles of short and long draws, which are drawn side by side and one after
the other: every member against the FP64 sum of its own draw (1e-5 sigma, the
grouped and the transform kernels' bound), and the grouped members against their
single runs bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from scarf3d_amd.hip import Hip
from srm_cases import init_product, structured_cfg

pytestmark = pytest.mark.gpu


def _members(longest):
    out = []
    for q in range(40):
        nharm = (150, 64, 700, 150, longest)[q % 5] + q
        out.append(dict(nd=3, fe=(30 + q, 28, 20 + q % 7), ds=25.0, acf=q % 2, cl=(150.0, 120.0, 100.0), sigma=0.05,
                        hurst=0.1 + 0.01 * q, nharm=nharm, seed=q + 1, rescale=int(q == 7)))
    return out


def _cfg(m, real):
    return structured_cfg(n=m["fe"], ds=m["ds"], acf=m["acf"], cl=m["cl"], sigma=m["sigma"], hurst=m["hurst"],
                          nharm=m["nharm"], rescale=m["rescale"], real=real)


@pytest.mark.parametrize("kernel,longest", [("auto", 400), ("auto", 20000), ("mfma_bf16x3", 5000)])
@pytest.mark.parametrize("flavour", ["f", "d"])
def test_members_of_short_and_long_draws(request, flavour, kernel, longest):
    lib = request.getfixturevalue("lib_" + flavour)
    hip = Hip()
    members = _members(longest)
    bufs = [hip.empty(int(np.prod(m["fe"])), lib.dtype) for m in members]
    print("[case]", flavour, kernel, longest, flush=True)
    lib.ensemble_execute(members, [b.ptr for b in bufs], kernel)
    worst = 0.0
    for q, (m, b) in enumerate(zip(members, bufs)):
        init_product(lib, _cfg(m, lib.dtype))
        d = hip.empty(int(np.prod(m["fe"])), np.float64)
        lib.srm_draw(m["seed"])
        lib.srm_run_fp64(d.ptr)
        lib.finalize()
        worst = max(worst, np.abs(b.numpy() - d.numpy()).max() / m["sigma"])
        d.free()
        if kernel != "auto" and q % 5 in (0, 4):
            init_product(lib, _cfg(m, lib.dtype))
            lib.set_kernel(kernel)
            single, _ = lib.execute(m["seed"])
            lib.set_kernel("auto")
            lib.finalize()
            assert np.array_equal(b.numpy(), single.reshape(-1, order="F")), q
    print(f"  max {worst:.2e} sigma", flush=True)
    for b in bufs:
        b.free()
    assert worst <= 1e-5
