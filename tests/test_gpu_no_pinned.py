"""A process that is refused pinned host memory gets the same fields
(tests/native/no_pinned.cpp)."""
import pytest

from native_lib import build_check, run_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flavour", ["f", "d"])
def test_without_pinned_memory_the_fields_are_the_same(tmp_path, flavour):
    exe = build_check("no_pinned", tmp_path, flavour)
    env = {"PATH": "/usr/bin:/bin", "SCARF_TUNE": "0"}
    a = run_check(exe, 1, env=env)
    b = run_check(exe, 0, env=env)
    print(a, flush=True)
    assert a == b and len(a.splitlines()) == 16
