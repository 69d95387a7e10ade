"""Point lists where their raw coordinates find no room on the device
(tests/native/points_upload.cpp)."""
import pytest

from native_lib import build_check, run_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flavour", ["f", "d"])
def test_coordinates_without_room_for_raw_ones(tmp_path, flavour):
    out = run_check(build_check("points_upload", tmp_path, flavour))
    print(out, flush=True)
    assert out.rstrip().endswith("0 bad")
