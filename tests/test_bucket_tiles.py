"""The bucket plan's tilings and its map from workgroups to tiles (runtime/bucket.h), on the CPU."""
from host_build import run_check


def test_tilings_and_shares(tmp_path):
    run_check("bucket_tiles_check", tmp_path)
