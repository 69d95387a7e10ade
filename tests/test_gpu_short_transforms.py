"""FIM's dense transform of short lines in float rounds no more than its bound
(tests/native/short_transforms.cpp)."""
import pytest

from native_lib import build_check, run_check

pytestmark = pytest.mark.gpu


def test_short_lines_round_within_their_bound(tmp_path):
    out = run_check(build_check("short_transforms", tmp_path))
    print(out, flush=True)
    assert out.rstrip().endswith("0 bad")
