"""The pool behind the bucket plan's and the local sort's device memory (runtime/workspace.h),
on the CPU with counted memory."""
from host_build import run_check


def test_pool(tmp_path):
    run_check("workspace_check", tmp_path)
