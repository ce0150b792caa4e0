"""The forward's tiles and the boundary slots of their re-runs (host code)."""
from native_check import run_check


def test_boundary_slots_over_rounds(tmp_path):
    run_check(tmp_path, "check_fw_plan")
