"""The run's status in pinned memory (runtime/run_status.h), on the CPU."""
from host_build import run_check


def test_stale_status_is_refused(tmp_path):
    run_check("run_status_check", tmp_path)
