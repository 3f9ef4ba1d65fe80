"""The batched point-to-point step at the edges of its list sizes: 256 pairs (small workgroups scan
the list), 4096 (one scan per CU), more (a scan kernel, tiles of 4096 pairs and, past 1024
tiles, of more), with empty runs, one pair that holds nearly everything, and any alignment."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(pkg, torch, sizes, seed, replay=0):
    rng = np.random.default_rng(seed)
    n = len(sizes)
    gap = rng.integers(0, 20, n)
    src = np.cumsum(sizes + gap) - sizes
    order = rng.permutation(n)
    dst = np.zeros(n, dtype=np.int64)
    dst[order] = np.cumsum((sizes + gap[::-1])[order]) - sizes[order]
    total = int(max((src + sizes).max(), (dst + sizes).max())) + 32
    send = torch.randint(0, 256, (total,), dtype=torch.uint8, device="cuda")
    recv = torch.full((total,), 0xAB, dtype=torch.uint8, device="cuda")
    pairs = torch.from_numpy(np.stack([src + send.data_ptr(), dst + recv.data_ptr(), sizes], axis=1).astype(np.int64)).cuda()
    plan = pkg.P2pPlan(n)
    if replay:
        plan.graph_replay(pairs.data_ptr(), n, replay)
    else:
        plan.execute(pairs.data_ptr(), n)
    torch.cuda.synchronize()
    plan.close()
    s, got = send.cpu().numpy(), recv.cpu().numpy()
    want = np.full(total, 0xAB, dtype=np.uint8)
    z = np.repeat(src - (np.cumsum(sizes) - sizes), sizes) + np.arange(int(sizes.sum()))
    w = np.repeat(dst - (np.cumsum(sizes) - sizes), sizes) + np.arange(int(sizes.sum()))
    want[w] = s[z]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 4095, 4096, 4097, 8193, 70001])
@pytest.mark.parametrize("kind", ["small", "empty_runs", "one_large"])
def test_list_sizes(n, kind, pkg, torch_gpu):
    print(f"[gpu] p2p list n={n} {kind}", flush=True)
    rng = np.random.default_rng(n)
    sizes = rng.integers(1, 200, n).astype(np.int64)
    if kind == "empty_runs":
        sizes[rng.random(n) < 0.7] = 0
        sizes[n // 3:2 * n // 3] = 0
    if kind == "one_large":
        sizes[n // 2] = (5 << 20) + 3
    run(pkg, torch_gpu, sizes, n, replay=2 if n % 2 else 0)


def test_more_than_1024_tiles(pkg, torch_gpu):
    """1024 * 4096 + 5 pairs: tiles of 8192."""
    n = 1024 * 4096 + 5
    print(f"[gpu] p2p list n={n}", flush=True)
    sizes = np.zeros(n, dtype=np.int64)
    sizes[::97] = np.arange(len(sizes[::97])) % 37
    sizes[-1] = 9000
    run(pkg, torch_gpu, sizes, 3)
