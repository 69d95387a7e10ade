"""Host-side rules of the device paths, at sizes no test could run: checked on
the CPU through the built library's internal headers."""
from native_lib import build_check, run_check


def test_point_lists_of_any_size_launch_within_the_limit(tmp_path):
    assert "0 bad" in run_check(build_check("points_launches", tmp_path))


def test_the_transforms_workspace_is_bounded(tmp_path):
    out = run_check(build_check("transform_plan_bounds", tmp_path))
    assert ", 0 bad" in out and int(out.split()[-4]) > 500, out


def test_an_ensembles_draws_take_the_faster_way(tmp_path):
    assert "0 bad" in run_check(build_check("draws_side_by_side", tmp_path))
