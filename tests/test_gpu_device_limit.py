"""Calls at SCARF_DEVICE_MEMORY_LIMIT: what is enough for the direct sums is
enough under auto too, in the first call and in later ones, and what the
library holds stays within it (tests/native/device_limit.cpp)."""
import pytest

from native_lib import build_check, run_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flavour", ["f", "d"])
def test_limits_hold_and_suffice(tmp_path, flavour):
    out = run_check(build_check("device_limit", tmp_path, flavour))
    print(out, flush=True)
    assert out.rstrip().endswith("0 bad")
