"""The batched reduction at the edges of its kernels' ranges: the staged fold's tiles and batches
of ranks, the last column that is not whole in every kernel, and sends that are also the
receive buffers.  Bit-exact with the oracle's rank-order fold."""
import numpy as np
import pytest

from oracle_py import reduce
from test_gpu_batched_reduce import MPI_DOUBLE, MPI_FLOAT, MPI_INT, MPI_INT64_T, OP_MIN, OP_SUM, _inputs, _run

pytestmark = pytest.mark.gpu


# floats: staged up to 512 KiB (64 ranks and fewer) or 256 KiB, then narrow, wide from 8 MiB;
# integers: staged up to 128 KiB, then split
@pytest.mark.parametrize("dt,P,n", [
    (MPI_FLOAT, 1, 1), (MPI_FLOAT, 2, 3), (MPI_FLOAT, 513, 2), (MPI_DOUBLE, 65, 1), (MPI_FLOAT, 257, 5),
    (MPI_FLOAT, 1024, 1003), (MPI_DOUBLE, 300, 8191), (MPI_FLOAT, 3, 131073), (MPI_FLOAT, 3, 131071),
    (MPI_DOUBLE, 70, 32769), (MPI_FLOAT, 66, 65538), (MPI_DOUBLE, 2, (1 << 20) + 1), (MPI_FLOAT, 2, (1 << 21) + 3),
    (MPI_INT, 260, 32767), (MPI_INT, 260, 32771), (MPI_INT, 3, 200001), (MPI_INT64_T, 600, 16385), (MPI_INT, 5, (1 << 21) + 1)])
def test_sizes_match_oracle(dt, P, n, pkg, oracle, torch_gpu):
    print(f"[gpu] reduce sizes dt={dt} P={P} n={n}", flush=True)
    op = OP_SUM if P % 2 else OP_MIN
    ins = _inputs(np.random.default_rng(P + n), dt, op, P, n)
    if np.issubdtype(ins[0].dtype, np.floating) and n > 2:
        ins[P // 2][0] = np.inf
        ins[0][1] = -np.inf
        ins[P - 1][n - 1] = np.finfo(ins[0].dtype).max
    rc, exp = reduce(oracle, dt, op, ins)
    assert rc == 0
    eb = exp.view(np.uint8)
    outs = _run(pkg, torch_gpu, ins, dt, op, -1)
    for r in sorted({0, 1 % P, P // 2, P - 1}):
        assert np.array_equal(outs[r], eb), ("allreduce", r)
    outs = _run(pkg, torch_gpu, ins, dt, op, P - 1, graph_steps=2)
    assert np.array_equal(outs[P - 1], eb)
    assert P == 1 or np.all(outs[0] == 0xAB)


@pytest.mark.parametrize("P,n", [(7, 1003), (200, 40001), (40, 70001)])
def test_in_place_allreduce(P, n, pkg, oracle, torch_gpu):
    """Every rank's receive buffer is its send buffer (one step: the next would fold the sums)."""
    torch = torch_gpu
    print(f"[gpu] reduce in place P={P} n={n}", flush=True)
    ins = _inputs(np.random.default_rng(n), MPI_FLOAT, OP_SUM, P, n)
    rc, exp = reduce(oracle, MPI_FLOAT, OP_SUM, ins)
    assert rc == 0
    bufs = [torch.from_numpy(x.copy()).cuda() for x in ins]
    ptrs = torch.tensor([b.data_ptr() for b in bufs], dtype=torch.int64, device="cuda")
    plan = pkg.ReducePlan(P, n, MPI_FLOAT, OP_SUM, -1, ptrs.data_ptr(), ptrs.data_ptr())
    plan.execute()
    torch.cuda.synchronize()
    plan.close()
    for r in (0, P // 2, P - 1):
        assert np.array_equal(bufs[r].cpu().numpy().view(np.uint32), exp.view(np.uint32)), r
