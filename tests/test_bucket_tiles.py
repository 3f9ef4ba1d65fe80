"""The bucket plan's map from workgroups to tiles (runtime/bucket.h), on the CPU."""
from host_build import run_check


def test_every_xcd_has_its_share(tmp_path):
    run_check("bucket_tiles_check", tmp_path)
