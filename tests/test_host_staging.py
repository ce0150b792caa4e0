"""Host side of copies and device memory, against a HIP runtime in host memory."""
from native_check import run_check


def test_batch_used_with_another_device_current(tmp_path):
    run_check(tmp_path, "check_batch_device", library=True)


def test_uploads_leave_what_lies_between(tmp_path):
    run_check(tmp_path, "check_uploader", library=True)


def test_staging_memory_not_available(tmp_path):
    run_check(tmp_path, "check_stage_pool", library=True)


def test_table_copy_that_fails(tmp_path):
    run_check(tmp_path, "check_table_error", library=True)


def test_server_estimate_covers_a_batch(tmp_path):
    run_check(tmp_path, "check_footprint", library=True)


def test_idle_device_memory_is_given_up(tmp_path):
    run_check(tmp_path, "check_pool_memory", library=True)
