"""Roundings of the fast transforms' kernel and phases, on the CPU
(tests/native/kaiser_bessel_roundings.cpp)."""
from native_lib import build_check, run_check


def test_kernel_and_phases_round_within_their_bounds(tmp_path):
    print(run_check(build_check("kaiser_bessel_roundings", tmp_path)))
