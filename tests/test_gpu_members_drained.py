"""Ensembles whose draw fails leave nothing in flight on the caller's fields
(tests/native/members_drained.cpp)."""
import pytest

from native_lib import build_check, run_check

pytestmark = pytest.mark.gpu


def test_nothing_is_left_in_flight(tmp_path):
    out = run_check(build_check("members_drained", tmp_path))
    print(out, flush=True)
    assert out.rstrip().endswith("0 bad")
