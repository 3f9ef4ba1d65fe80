"""The split sort's work items up to parts of 2^32 - 1 keys (runtime/bucket.h), on the CPU."""
from host_build import run_check


def test_items_cover_their_part(tmp_path):
    run_check("sort_items_check", tmp_path)
