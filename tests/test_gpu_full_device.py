"""Workspaces of earlier calls make room for an ensemble's buffers, a tile
timing's and an FFT plan's (tests/native/full_device.cpp)."""
import pytest

from native_lib import build_check, run_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flavour", ["f", "d"])
def test_on_a_full_device_the_fields_are_the_same(tmp_path, flavour):
    exe = build_check("full_device", tmp_path, flavour)
    env = {"PATH": "/usr/bin:/bin"}
    a = run_check(exe, 1, env=env)
    b = run_check(exe, 0, env=env)
    print(a, flush=True)
    assert a == b and len(a.splitlines()) == (8 if flavour == "f" else 6)
