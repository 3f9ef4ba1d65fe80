"""The rank grid's MPI_Reduce / MPI_Allreduce around the slices of up to 16 elements per rank (4, 8
or 16 elements, ranks past the last multiple of a load, counts on both sides of the rule),
bit for bit against the oracle's rank-order fold.  Types of 1 to 16 bytes and user operators
go through t_op_table (test_gpu_runtime_programs.py)."""
import numpy as np
import pytest

from oracle_py import reduce

pytestmark = pytest.mark.gpu
TYPES = {2: np.int32, 13: np.float64}


@pytest.mark.parametrize("dt", [2, 13])
@pytest.mark.parametrize("P", [2, 5, 64, 67, 130])
def test_small_slices(P, dt, pkg, oracle, torch_gpu):
    from dphpc_project_amd import programs as pr
    torch = torch_gpu
    rng = np.random.default_rng(P * 100 + dt)
    with pkg.Runtime(P, heap_bytes=64 << 20, timeout_s=20.0) as rt:
        for n in sorted({1, 3, 4, 5, 4 * P, 4 * P + 1, 8 * P + 3, 16 * P - 1, 16 * P, 16 * P + 1}):
            x = rng.normal(size=(P, n)) if dt == 13 else rng.integers(-(1 << 20), 1 << 20, (P, n))
            x = x.astype(TYPES[dt])
            _, exp = reduce(oracle, dt, 2, [x[r] for r in range(P)])      # MPI_SUM
            d = torch.from_numpy(x).cuda()
            sec = torch.zeros(P, dtype=torch.float64, device="cuda")
            for kind, root in (("allreduce", 0), ("reduce", P - 1)):
                print(f"[gpu] rank {kind} P={P} n={n} dt={dt}", flush=True)
                out = torch.full((P, n + 4), -3, dtype=d.dtype, device="cuda")
                es = x.itemsize
                rt.run("coll", pr.CollArgs(0, pr.COLL_KINDS[kind], dt, 0, root, n, 2, 0, d.data_ptr(), out.data_ptr(),
                                           n * es, (n + 4) * es, sec.data_ptr(), 1))
                got = out.cpu().numpy()
                for r in range(P):
                    if kind == "allreduce" or r == root:
                        assert got[r, :n].tobytes() == exp.tobytes(), (kind, n, r)
                    else:
                        assert np.all(got[r] == -3), (kind, n, r)
                assert np.all(got[:, n:] == -3)
