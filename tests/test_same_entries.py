"""The traceback's same-branch transition entries against the forward's planes
(host code: the preparation of internal threading)."""
from native_check import run_check


def test_same_entries_of_internal_blocks(tmp_path):
    run_check(tmp_path, "check_same_entry", library=True)
