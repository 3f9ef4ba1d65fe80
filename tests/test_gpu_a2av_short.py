"""The batched Alltoallv around the rules that choose a row's copy loop (average segment, element
size, row size, windows of 512 segments) and at the rows' ends, against the oracle, bit for
bit: single steps, deferred mode and pipelined graphs."""
import numpy as np
import pytest

from oracle_py import alltoallv
from test_gpu_a2av import run_exchange

pytestmark = pytest.mark.gpu


def layout(rng, P, elem, mean, empty, hot):
    counts = rng.poisson(mean, (P, P)).astype(np.int32)
    counts[rng.random((P, P)) < empty] = 0
    if hot:
        counts[:, 1 % P] *= 40                      # one long row among short ones
        counts[2 % P, :] = 0
    if P > 600:
        counts[30:30 + 560, 5] = 0                  # more empty segments in a row than a window holds
    sdispls = np.zeros_like(counts)
    for s in range(P):
        gaps = rng.integers(0, 3, P)
        sdispls[s] = np.cumsum(counts[s] + gaps) - counts[s]
    sizes = [int((sdispls[s] + counts[s]).max()) for s in range(P)]
    send = [rng.integers(0, 256, max(1, n) * elem, dtype=np.uint8) for n in sizes]
    return send, counts, sdispls


@pytest.mark.parametrize("tune,graph", [(None, 0), ((0, -1, 2, 0, 1, 0), 0), ((0, 1, 8, 1, 4, 0), 0), ((0, -1, 0, -1, 0, 1), 0),
                                        (None, 3)])
@pytest.mark.parametrize("P,elem,mean,empty,hot", [
    (4, 4, 500, 0.0, False), (4, 8, 260, 0.0, True), (33, 4, 111, 0.1, True), (33, 1, 450, 0.1, True), (5, 1, 33000, 0.2, False),
    (2, 4, 70001, 0.0, False), (64, 3, 9, 0.5, False), (700, 1, 2, 0.4, False), (1, 1, 9000, 0.0, False)])
def test_row_kinds(P, elem, mean, empty, hot, tune, graph, pkg, oracle, torch_gpu):
    print(f"[gpu] a2av rows P={P} elem={elem} mean={mean} hot={hot} tune={tune} graph={graph}", flush=True)
    rng = np.random.default_rng(P * 77 + mean)
    send, counts, sdispls = layout(rng, P, elem, mean, empty, hot)
    offsets = [int(x) for x in rng.integers(0, 16, P)]
    got, rc, rd, nbytes = run_exchange(pkg, torch_gpu, send, counts, sdispls, elem, offsets=offsets, tune=tune,
                                       graph_steps=graph)
    exp, erc, erd = alltoallv(oracle, send, counts, sdispls, elem, counts.sum(axis=0))
    assert nbytes == int(counts.sum()) * elem
    assert np.array_equal(rc, erc) and np.array_equal(rd, erd)
    for d in range(P):
        assert np.array_equal(got[d], exp[d][:got[d].size]), f"rank {d}"
