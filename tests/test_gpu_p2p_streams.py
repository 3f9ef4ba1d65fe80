"""Point-to-point steps large enough to load (48 MiB) and to store (512 MiB) past the caches, by
each of the three copy kernels, with pairs at any alignment: equal bytes, and nothing outside
the pairs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mib", [70, 600])
@pytest.mark.parametrize("n", [3, 300, 5000])
def test_large_steps(n, mib, pkg, torch_gpu):
    torch = torch_gpu
    print(f"[gpu] p2p step of {mib} MiB, {n} pairs", flush=True)
    rng = np.random.default_rng(n)
    each = (mib << 20) // n
    sizes = each - rng.integers(0, 100, n)
    off = 16 + np.arange(n) * (each + 40) + rng.integers(0, 16, n)
    to = 16 + rng.permutation(n) * (each + 40) + rng.integers(0, 16, n)
    total = int(n * (each + 40) + 64)
    send = torch.randint(0, 255, (total,), dtype=torch.uint8, device="cuda")
    recv = torch.full((total,), 255, dtype=torch.uint8, device="cuda")
    want = recv.clone()
    for a, b, c in zip(off, to, sizes):
        want[b:b + c] = send[a:a + c]
    pairs = torch.from_numpy(np.stack([off + send.data_ptr(), to + recv.data_ptr(), sizes], axis=1).astype(np.int64)).cuda()
    plan = pkg.P2pPlan(n)
    plan.execute(pairs.data_ptr(), n)
    torch.cuda.synchronize()
    plan.close()
    assert torch.equal(recv, want)
