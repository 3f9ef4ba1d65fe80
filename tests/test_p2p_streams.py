"""What a point-to-point step leaves in the caches (runtime/batched_p2p.h), on the CPU."""
from host_build import run_check


def test_rule_goes_by_bytes(tmp_path):
    run_check("p2p_streams_check", tmp_path)
