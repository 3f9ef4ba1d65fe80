"""The bucket plan's and the local sort's kernels at the edges of their tiles and dispatch
rules, against the oracle's bucket plan and numpy.sort (whole numbers: equal, no tolerance)."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from oracle_py import bucket_plan

pytestmark = pytest.mark.gpu


def make_keys(rng, kind, shape, key_bits):
    top = 1 << key_bits
    if kind == "equal":
        return np.full(shape, top - 1, dtype=np.uint32)
    if kind == "skewed":     # most keys in one bucket (part), the rest anywhere
        k = rng.integers(0, top, shape, dtype=np.uint32)
        return np.where(rng.random(shape) < 0.9, k % max(1, top >> 9), k).astype(np.uint32)
    if kind == "sorted":
        return np.sort(rng.integers(0, top, shape, dtype=np.uint32).reshape(-1)).reshape(shape)
    return rng.integers(0, top, shape, dtype=np.uint32)


# tiles of 4096 and 16384 keys (up to 1024 buckets), 2048 and 8192 (more); 8 ranks per group of
# workgroups; up to 64 ranks the splitters' workgroup sums the columns
@pytest.mark.parametrize("kind", ["uniform", "skewed", "equal", "sorted"])
@pytest.mark.parametrize("P,n,key_bits,bucket_bits", [
    (1, 1, 1, 1), (2, 64, 5, 3), (3, 4095, 11, 9), (8, 4097, 16, 10), (9, 2049, 13, 11), (64, 1000, 12, 12),
    (65, 777, 20, 10), (130, 63, 23, 9), (513, 16385, 18, 10), (300, 8193, 17, 12)])
def test_bucket_plan_edges(P, n, key_bits, bucket_bits, kind, pkg, oracle, torch_gpu):
    torch = torch_gpu
    print(f"[gpu] bucket_plan P={P} n={n} bits={key_bits}/{bucket_bits} {kind}", flush=True)
    keys = make_keys(np.random.default_rng(P + n), kind, (P, n), key_bits)
    d = torch.from_numpy(keys.view(np.int32)).cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    kb1 = torch.full((P * n + 64,), -1, **i32)
    sc, sd = torch.full((P, P), -1, **i32), torch.full((P, P), -1, **i32)
    lo, hi = torch.full((P,), -1, **i32), torch.full((P,), -1, **i32)
    pkg.bucket_plan(d.data_ptr(), P, n, key_bits, bucket_bits, kb1.data_ptr(), sc.data_ptr(), sd.data_ptr(),
                    lo.data_ptr(), hi.data_ptr())
    e_kb1, e_sc, e_sd, e_lo, e_hi = bucket_plan(oracle, keys, key_bits, bucket_bits)
    got = kb1.cpu().numpy()
    assert np.array_equal(got[:P * n].view(np.uint32), np.asarray(e_kb1).reshape(-1).view(np.uint32))
    assert np.all(got[P * n:] == -1)
    assert np.array_equal(lo.cpu().numpy(), e_lo) and np.array_equal(hi.cpu().numpy(), e_hi)
    assert np.array_equal(sc.cpu().numpy(), e_sc) and np.array_equal(sd.cpu().numpy(), e_sd)


# more than one tile per workgroup (tables past 32 MiB): two per workgroup, and a rank's only
# workgroup, whose counts become the prefix in place
@pytest.mark.parametrize("kind", ["uniform", "skewed"])
@pytest.mark.parametrize("P,n,key_bits,bucket_bits", [(3, 6000000, 23, 12), (1100, 8193, 17, 12)])
def test_bucket_plan_tiles_in_turn(P, n, key_bits, bucket_bits, kind, pkg, oracle, torch_gpu):
    test_bucket_plan_edges(P, n, key_bits, bucket_bits, kind, pkg, oracle, torch_gpu)


def test_bucket_plan_without_a_table(torch_gpu):
    """The tiling for the case that memory for the table is not to be had (tests/programs/bucket_turns.hip)."""
    exe = os.path.join(ROOT, "tests", "programs", "_build", "bucket_turns")
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and "all equal" in res.stdout, res.stdout + res.stderr


# one table up to 14 bits, parts of 2^14 values up to 24, counters in HBM beyond and when the
# output overlaps the keys; tiles of 16384 keys; large parts are shared by workgroups
@pytest.mark.parametrize("kind", ["uniform", "skewed", "equal", "sorted"])
@pytest.mark.parametrize("n,key_bits,shift,in_place", [
    (0, 9, 0, False), (1, 1, 1, False), (5, 14, 1, False), (16385, 11, 3, False), (600001, 14, 0, False), (1, 15, 0, False),
    (16383, 15, 1, False), (16385, 20, 2, False), (300007, 16, 1, False), (2000003, 23, 3, False), (70001, 24, 0, False),
    (70001, 25, 1, False), (50001, 12, 0, True), (50001, 18, 1, True)])
def test_local_sort_edges(n, key_bits, shift, in_place, kind, pkg, torch_gpu):
    torch = torch_gpu
    print(f"[gpu] local_sort n={n} bits={key_bits} shift={shift} in_place={in_place} {kind}", flush=True)
    keys = make_keys(np.random.default_rng(n + key_bits), kind, n, key_bits)
    d = torch.zeros(n + 40, dtype=torch.int32, device="cuda")
    d[shift:shift + n] = torch.from_numpy(keys.view(np.int32)).cuda()
    out = d if in_place else torch.full((n + 40,), -1, dtype=torch.int32, device="cuda")
    at = shift if in_place else 3 - shift      # keys and output on different 16-byte phases
    before = out.cpu().numpy()
    pkg.local_sort(d.data_ptr() + 4 * shift, n, key_bits, out.data_ptr() + 4 * at)
    got = out.cpu().numpy()
    assert np.array_equal(got[at:at + n].view(np.uint32), np.sort(keys))
    assert np.array_equal(got[:at], before[:at]) and np.array_equal(got[at + n:], before[at + n:])


def test_workspaces_are_given_back(pkg, torch_gpu):
    """What bucket_plan and local_sort keep idle between calls is bounded and can be given back."""
    torch = torch_gpu
    pkg.workspace_trim()
    free0 = torch.cuda.mem_get_info()[0]
    x = torch.randint(0, 1 << 20, (1 << 22,), dtype=torch.int32, device="cuda")
    y = torch.empty_like(x)
    for n in (1 << 12, 1 << 18, 1 << 22):
        pkg.local_sort(x.data_ptr(), n, 20, y.data_ptr())
    del x, y
    torch.cuda.empty_cache()
    assert free0 - torch.cuda.mem_get_info()[0] <= 72 << 20
    pkg.workspace_trim()
    assert free0 - torch.cuda.mem_get_info()[0] <= 8 << 20
