"""A run on the rank grid after some other HIP call of the thread has failed (its error is the
caller's, who may not have asked for it yet): the run's own calls succeed, so the run does."""
import pytest

pytestmark = pytest.mark.gpu


def test_run_after_a_refused_call(pkg, torch_gpu):
    from dphpc_project_amd import programs as pr
    torch = torch_gpu
    print("[gpu] run after a refused hipSetDevice", flush=True)
    P, n = 4, 33
    d = torch.arange(P * n, dtype=torch.int32, device="cuda").reshape(P, n)
    out = torch.zeros_like(d)
    sec = torch.zeros(P, dtype=torch.float64, device="cuda")
    with pkg.Runtime(P, heap_bytes=64 << 20, timeout_s=20.0) as rt:
        assert pkg.load_library().hipSetDevice(12345) != 0
        try:
            rt.run("coll", pr.CollArgs(0, pr.COLL_KINDS["allreduce"], 2, 0, 0, n, 2, 0, d.data_ptr(), out.data_ptr(),
                                       4 * n, 4 * n, sec.data_ptr(), 1))
        finally:
            pkg.load_library().hipGetLastError()
        assert torch.equal(out, d.sum(0, dtype=torch.int32).expand(P, n))
