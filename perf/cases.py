"""The work whose speed matters to a user of this framework, as cases that can be measured.

A case is a dict of plain values; `op` names the path:

  alltoallv   one step's uneven MPI_Alltoallv over all ranks (A2avPlan), single steps or a
              graph of steps, as the exchange of a bucket sort, of tokens or of ragged rows
  reduce      one step's MPI_Reduce / MPI_Allreduce over all ranks (ReducePlan)
  p2p         one step's matched Send/Recv pairs (P2pPlan)
  particles   two steps of the particle exchange on a periodic rank grid (ParticlePlan)
  bucket_sort a distributed integer bucket sort: bucket plan, exchange, local sort
  coll        a rank program that makes ten calls of one collective (Runtime, "coll")
  pingpong    a rank program of ping-pong or ring messages (Runtime, "p2p")

Inputs come from the seed alone.  Everything here is bytes, integers or reductions in a
fixed (rank) order, so results are the same bits on any correct implementation."""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "dphpc-project_amd")

TORCH_TYPES = {"int32": torch.int32, "int64": torch.int64, "float32": torch.float32, "float64": torch.float64}
MPI_TYPES = {"int32": "MPI_INT", "int64": "MPI_INT64_T", "float32": "MPI_FLOAT", "float64": "MPI_DOUBLE"}
OPS = {"max": 0, "min": 1, "sum": 2}
COLL_CALLS = 10
PING_ITERS = 20


def package():
    """The framework's Python package (its folder's name is no module name)."""
    name = "dphpc_project_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(PACKAGE, "__init__.py"), submodule_search_locations=[PACKAGE])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def listed():
    return [
        # a step of a small job: 16 ranks, a few dozen doubles per pair; launches and latency
        {"name": "alltoallv_small", "op": "alltoallv", "ranks": 16, "elem": 8, "bytes": 48 << 10, "skew": 0.0, "steps": 1},
        # tokens or rows of uneven sizes, byte-granular, some receivers much hotter: one step
        {"name": "alltoallv_skewed", "op": "alltoallv", "ranks": 200, "elem": 1, "bytes": (48 << 20) + 77, "skew": 1.1,
         "steps": 1},
        # the bucket-sort exchange: 512 ranks x 1 MiB of uint32 keys, ten steps per graph
        {"name": "alltoallv_keys", "op": "alltoallv", "ranks": 512, "elem": 4, "bytes": 512 << 20, "skew": 0.0,
         "steps": 10},
        # a short vector of scalars reduced to one rank
        {"name": "reduce_small", "op": "reduce", "ranks": 32, "count": 1003, "dtype": "float32", "fold": "sum", "root": 5},
        # the batched Allreduce of 1024 ranks x 1 MiB of doubles
        {"name": "allreduce_large", "op": "reduce", "ranks": 1024, "count": 131072, "dtype": "float64", "fold": "sum",
         "root": -1},
        # face messages of an 8x8x8 rank grid: 3072 uneven pairs of some KiB
        {"name": "p2p_faces", "op": "p2p", "pairs": 3072, "bytes": 15 << 20, "grain": 8},
        # long messages: 64 pairs of about 16 MiB
        {"name": "p2p_long", "op": "p2p", "pairs": 64, "bytes": (1 << 30) + 12, "grain": 4},
        # the particle exchange at its full size: 2^24 particles on 8x8x8 ranks, two steps
        {"name": "particles_full", "op": "particles", "gx": 8, "gy": 8, "gz": 8, "n0": 32768, "mode": 0},
        # integer sort at NPB class S: 2^16 keys on 4 ranks
        {"name": "bucket_sort_small", "op": "bucket_sort", "ranks": 4, "n": 16384, "key_bits": 11, "bucket_bits": 9,
         "dist": "npb"},
        # integer sort of 2^27 uniform keys below 2^23 on 512 ranks (NPB class C's sizes)
        {"name": "bucket_sort_large", "op": "bucket_sort", "ranks": 512, "n": 1 << 18, "key_bits": 23,
         "bucket_bits": 10, "dist": "uniform"},
        # a rank program's collective in its usual range: Allreduce of 1000 doubles on 256 ranks
        {"name": "rank_allreduce", "op": "coll", "ranks": 256, "kind": "allreduce", "count": 1000, "dtype": "float64"},
        # ping-pong of 4 KiB messages, blocking Send/Recv, 256 ranks
        {"name": "rank_pingpong", "op": "pingpong", "ranks": 256, "bytes": 4096, "mode": 0},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["alltoallv", "alltoallv", "reduce", "reduce", "p2p", "p2p", "particles", "bucket_sort",
                     "bucket_sort", "coll", "pingpong"])
    if op == "alltoallv":
        ranks = _log(rng, 4, 512)
        return {"op": op, "ranks": ranks, "elem": rng.choice([1, 4, 4, 8]),
                "bytes": _log(rng, max(16 << 10, 16 * ranks * ranks), 512 << 20),
                "skew": rng.choice([0.0, 0.0, 0.6, 1.1]), "steps": rng.choice([1, 1, 10])}
    if op == "reduce":
        ranks = _log(rng, 2, 1024)
        dtype = rng.choice(["float32", "float64", "float64", "int32", "int64"])
        size = torch.empty(0, dtype=TORCH_TYPES[dtype]).element_size()
        count = _log(rng, 16, min(1 << 22, (1 << 30) // (ranks * size)))
        return {"op": op, "ranks": ranks, "count": count, "dtype": dtype, "fold": rng.choice(["sum", "sum", "max", "min"]),
                "root": rng.choice([-1, rng.randrange(ranks)])}
    if op == "p2p":
        pairs = _log(rng, 2, 65536)
        return {"op": op, "pairs": pairs, "bytes": _log(rng, max(4096, 64 * pairs), 1 << 30), "grain": rng.choice([1, 4, 8])}
    if op == "particles":
        g = [rng.choice([1, 2, 3, 4, 5, 8]) for _ in range(3)]
        return {"op": op, "gx": g[0], "gy": g[1], "gz": g[2], "n0": _log(rng, 200, 32768), "mode": rng.choice([0, 0, 1])}
    if op == "bucket_sort":
        ranks = _log(rng, 4, 512)
        key_bits = rng.randint(11, 23)
        return {"op": op, "ranks": ranks, "n": _log(rng, 1024, 1 << 18), "key_bits": key_bits,
                "bucket_bits": rng.choice([9, 10]), "dist": rng.choice(["uniform", "npb", "zipf"])}
    if op == "coll":
        ranks = _log(rng, 8, 512)
        kind = rng.choice(["bcast", "reduce", "allreduce", "alltoall", "allgather"])
        most = 1 << 16 if kind != "allgather" else max(1, (1 << 22) // ranks)
        count = _log(rng, 1, most)
        if kind == "alltoall":
            count = max(1, count // ranks) * ranks
        return {"op": op, "ranks": ranks, "kind": kind, "count": count, "dtype": rng.choice(["int32", "float64"])}
    return {"op": op, "ranks": 2 * _log(rng, 1, 256), "bytes": _log(rng, 8, 1 << 20), "mode": rng.randrange(4)}


class State:
    """What a program keeps between calls: tensors and plans, by attribute."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _int64s(values):
    return torch.tensor([int(v) for v in values], dtype=torch.int64, device="cuda")


# ------------------------------------------------------------------ alltoallv
def _a2av_counts(case, seed):
    """send counts [P][P] in elements: each rank's elements dealt over the destinations, whose
    popularity falls as 1 / k^skew in an order drawn from the seed."""
    rng = np.random.default_rng(seed)
    P, total = case["ranks"], case["bytes"] // case["elem"]
    w = np.arange(1, P + 1, dtype=np.float64) ** -case["skew"]
    w = rng.permutation(w / w.sum())
    each = np.full(P, total // P)
    each[: total % P] += 1
    return rng.multinomial(each, w).astype(np.int64)


def _a2av_inputs(case, seed):
    counts = _a2av_counts(case, seed)
    n = int(counts.sum()) * case["elem"]
    send = torch.randint(0, 256, (max(n, 1),), dtype=torch.uint8, device="cuda", generator=_gen(seed))
    return counts, send


def _prepare_alltoallv(case, seed):
    pkg, P, e = package(), case["ranks"], case["elem"]
    counts, send = _a2av_inputs(case, seed)
    displs = np.cumsum(counts, axis=1) - counts
    first = np.cumsum(counts.sum(axis=1)) - counts.sum(axis=1)
    rtot = counts.sum(axis=0)
    roff = np.cumsum(rtot) - rtot
    recv = torch.zeros(send.numel(), dtype=torch.uint8, device="cuda")
    s = State(send=send, recv=recv, steps=case["steps"],
              sc=torch.from_numpy(counts.astype(np.int32)).cuda(), sd=torch.from_numpy(displs.astype(np.int32)).cuda(),
              rc=torch.zeros((P, P), dtype=torch.int32, device="cuda"),
              rd=torch.zeros((P, P), dtype=torch.int32, device="cuda"),
              sptr=_int64s(send.data_ptr() + e * first), rptr=_int64s(recv.data_ptr() + e * roff))
    s.plan = pkg.A2avPlan(P, e, s.sptr.data_ptr(), s.sc.data_ptr(), s.sd.data_ptr(), s.rptr.data_ptr(),
                          s.rc.data_ptr(), s.rd.data_ptr())
    return s


def _run_alltoallv(s):
    stream = torch.cuda.current_stream().cuda_stream
    if s.steps == 1:
        s.plan.execute(stream)
    else:
        s.plan.graph_replay(s.steps, stream)
    return {"recv": s.recv, "recv_counts": s.rc, "recv_displs": s.rd}


def _exchanged(counts, send, elem):
    """The receive buffers, one after the other, of dense send buffers in rank order."""
    c = torch.from_numpy(counts).cuda()
    flat = c.reshape(-1)
    src = (flat.cumsum(0) - flat).reshape(c.shape).t().reshape(-1)      # where (s, d) starts, in (d, s) order
    ct = c.t().reshape(-1)
    n = int(ct.sum())
    idx = torch.repeat_interleave(src - (ct.cumsum(0) - ct), ct) + torch.arange(n, device="cuda")
    rows = send[: n * elem].reshape(n, elem)
    return rows[idx].reshape(-1)


def _exact_alltoallv(case, seed):
    counts, send = _a2av_inputs(case, seed)
    ct = torch.from_numpy(np.ascontiguousarray(counts.T)).cuda()
    return {"recv": _exchanged(counts, send, case["elem"]), "recv_counts": ct, "recv_displs": ct.cumsum(1) - ct}


# ------------------------------------------------------------------ reduce
def _reduce_input(case, seed):
    """[P][row]: the rank buffers, each row padded to whole 256-byte blocks like an allocation."""
    t = TORCH_TYPES[case["dtype"]]
    size = torch.empty(0, dtype=t).element_size()
    row = -(-case["count"] * size // 256) * 256 // size
    shape, g = (case["ranks"], row), _gen(seed)
    if t.is_floating_point:
        return torch.randn(shape, dtype=t, device="cuda", generator=g)
    return torch.randint(-(1 << 20), (1 << 20) + 1, shape, dtype=t, device="cuda", generator=g)


def _prepare_reduce(case, seed):
    pkg, P, root = package(), case["ranks"], case["root"]
    x = _reduce_input(case, seed)
    step = x.stride(0) * x.element_size()
    y = torch.zeros((P if root < 0 else 1, x.shape[1]), dtype=x.dtype, device="cuda")
    to = [y.data_ptr() + (r * step if root < 0 else 0) for r in range(P)]
    s = State(x=x, y=y, count=case["count"], sptr=_int64s(x.data_ptr() + r * step for r in range(P)), rptr=_int64s(to))
    s.plan = pkg.ReducePlan(P, case["count"], pkg.DT[MPI_TYPES[case["dtype"]]], OPS[case["fold"]], root,
                            s.sptr.data_ptr(), s.rptr.data_ptr())
    return s


def _run_reduce(s):
    s.plan.execute(torch.cuda.current_stream().cuda_stream)
    return s.y[:, :s.count]


def _exact_reduce(case, seed):
    x = _reduce_input(case, seed)[:, :case["count"]]
    wide = torch.float64 if x.dtype.is_floating_point else torch.int64
    acc = x[0].to(wide)
    for r in range(1, case["ranks"]):
        v = x[r].to(wide)
        acc = acc + v if case["fold"] == "sum" else torch.maximum(acc, v) if case["fold"] == "max" else torch.minimum(acc, v)
    return acc.expand(case["ranks"] if case["root"] < 0 else 1, -1)


# ------------------------------------------------------------------ p2p
def _p2p_inputs(case, seed):
    """Pair sizes (log-normal around their mean, in whole grains, some empty) and the bytes."""
    rng = np.random.default_rng(seed)
    w = rng.lognormal(0.0, 0.6, case["pairs"])
    w[rng.random(case["pairs"]) < 0.01] = 0.0
    w[0] = max(w[0], 0.1)
    sizes = (w / w.sum() * (case["bytes"] // case["grain"])).astype(np.int64) * case["grain"]
    sizes[0] += case["bytes"] // case["grain"] * case["grain"] - int(sizes.sum())
    order = rng.permutation(case["pairs"])       # where each pair's bytes lie in the receive buffer
    send = torch.randint(0, 256, (int(sizes.sum()),), dtype=torch.uint8, device="cuda", generator=_gen(seed))
    return sizes, order, send


def _p2p_offsets(sizes, order):
    src = np.cumsum(sizes) - sizes
    dst = np.zeros_like(sizes)
    dst[order] = np.cumsum(sizes[order]) - sizes[order]
    return src, dst


def _prepare_p2p(case, seed):
    sizes, order, send = _p2p_inputs(case, seed)
    src, dst = _p2p_offsets(sizes, order)
    recv = torch.zeros_like(send)
    table = np.stack([src + send.data_ptr(), dst + recv.data_ptr(), sizes], axis=1)
    return State(send=send, recv=recv, n=case["pairs"], pairs=torch.from_numpy(table).cuda(),
                 plan=package().P2pPlan(case["pairs"]))


def _run_p2p(s):
    s.plan.execute(s.pairs.data_ptr(), s.n, torch.cuda.current_stream().cuda_stream)
    return s.recv


def _exact_p2p(case, seed):
    sizes, order, send = _p2p_inputs(case, seed)
    src, _ = _p2p_offsets(sizes, order)
    n = torch.from_numpy(sizes[order]).cuda()
    base = torch.from_numpy(src[order]).cuda() - (n.cumsum(0) - n)
    return send[torch.repeat_interleave(base, n) + torch.arange(send.numel(), device="cuda")]


# ------------------------------------------------------------------ particles
def _particle_inputs(case, seed):
    """States [P][cap][8] with a little under n0 to n0 particles per rank, ids 0, 1, ..."""
    g = (case["gx"], case["gy"], case["gz"])
    P, n0 = g[0] * g[1] * g[2], case["n0"]
    cap = n0 + n0 // 3 + 256
    rng = np.random.default_rng(seed)
    counts = torch.from_numpy(rng.integers(n0 - n0 // 16, n0 + 1, P)).cuda()
    parts = torch.rand((P, cap, 8), dtype=torch.float64, device="cuda", generator=_gen(seed))
    r = torch.arange(P, device="cuda")
    parts[:, :, 0] += (r % g[0])[:, None]
    parts[:, :, 1] += (r // g[0] % g[1])[:, None]
    parts[:, :, 2] += (r // (g[0] * g[1]))[:, None]
    parts[:, :, 7] = (counts.cumsum(0) - counts)[:, None] + torch.arange(cap, device="cuda")
    return g, cap, parts, counts


def _prepare_particles(case, seed):
    g, cap, parts, counts = _particle_inputs(case, seed)
    s = State(a=parts, ca=counts, b=torch.zeros_like(parts), cb=torch.zeros_like(counts),
              plan=package().ParticlePlan(g, cap, int(seed)))
    s.plan.exchange_mode(case["mode"])
    s.plan.prepare(s.a.data_ptr(), s.ca.data_ptr(), 0, torch.cuda.current_stream().cuda_stream)
    return s


def _run_particles(s):
    stream = torch.cuda.current_stream().cuda_stream
    a, b = (s.a.data_ptr(), s.ca.data_ptr()), (s.b.data_ptr(), s.cb.data_ptr())
    s.plan.step(*a, *b, stream)
    s.plan.step(*b, *a, stream)
    return {"parts": s.a, "counts": s.ca}


def _philox(c, key):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors that hold 32-bit words."""
    low, (x, y, z, w), (k0, k1) = 0xFFFFFFFF, c, key
    for i in range(10):
        if i:
            k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
        p, q = x * 0xD2511F53, z * 0xCD9E8D57            # the products' low 64 bits
        x, y, z, w = ((q >> 32) & low) ^ y ^ k0, q & low, ((p >> 32) & low) ^ w ^ k1, p & low
    return x, y


def _particle_step(g, parts, counts, seed, step, out):
    """One step on torch: stayers first, then the arrivals by source rank and order, into `out`."""
    P, cap = parts.shape[:2]
    live = torch.arange(cap, device="cuda")[None, :] < counts[:, None]
    rank = torch.arange(P, device="cuda")[:, None].expand(P, cap)[live]
    v = parts[live]
    ids = v[:, 7].to(torch.int64)
    x, y = _philox((ids & 0xFFFFFFFF, ids >> 32, torch.full_like(ids, step), torch.full_like(ids, 0x0B17E505)),
                   (seed & 0xFFFFFFFF, seed >> 32))
    moves, d = x < 214748365, (y * 6) >> 32
    at = [rank % g[0], rank // g[0] % g[1], rank // (g[0] * g[1])]
    for axis in range(3):
        by = torch.where(moves & (d // 2 == axis), 1 - 2 * (d % 2), torch.zeros_like(d))
        at[axis] = (at[axis] + by) % g[axis]
        u = v[:, axis] + by.to(torch.float64)
        u = torch.where((by != 0) & (u >= g[axis]), u - g[axis], u)
        v[:, axis] = torch.where((by != 0) & (u < 0), u + g[axis], u)
    to = at[0] + g[0] * (at[1] + g[1] * at[2])
    order = torch.sort((to * 2 + moves.to(torch.int64)) * P + rank, stable=True).indices
    to = to[order]
    new = torch.bincount(to, minlength=P)
    slot = torch.arange(to.numel(), device="cuda") - (new.cumsum(0) - new)[to]
    out[to, slot] = v[order]
    return out, new


def _exact_particles(case, seed):
    g, cap, a, counts = _particle_inputs(case, seed)
    b, between = _particle_step(g, a, counts, int(seed), 0, torch.zeros_like(a))
    a, after = _particle_step(g, b, between, int(seed), 1, a)
    return {"parts": a, "counts": after}


# ------------------------------------------------------------------ bucket sort
def _keys(case, seed):
    n, top, g = case["ranks"] * case["n"], 1 << case["key_bits"], _gen(seed)
    if case["dist"] == "uniform":
        return torch.randint(0, top, (n,), dtype=torch.int32, device="cuda", generator=g)
    if case["dist"] == "npb":       # NPB IS: the mean of four uniform draws
        k = torch.zeros(n, dtype=torch.int32, device="cuda")
        for _ in range(4):
            k += torch.randint(0, top, (n,), dtype=torch.int32, device="cuda", generator=g)
        return k >> 2
    w = torch.arange(1, top + 1, dtype=torch.float64, device="cuda") ** -1.1
    cdf = w.cumsum(0)
    u = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
    return torch.searchsorted(cdf / cdf[-1], u, right=True).clamp_(max=top - 1).to(torch.int32)


def _prepare_bucket_sort(case, seed):
    pkg, P, n = package(), case["ranks"], case["n"]
    i32 = dict(dtype=torch.int32, device="cuda")
    s = State(P=P, n=n, key_bits=case["key_bits"], bucket_bits=case["bucket_bits"], keys=_keys(case, seed),
              sent=torch.zeros(P * n, **i32), recv=torch.zeros(P * n + 64, **i32), out=torch.zeros(P * n, **i32),
              sc=torch.zeros((P, P), **i32), sd=torch.zeros((P, P), **i32), rc=torch.zeros((P, P), **i32),
              rd=torch.zeros((P, P), **i32), lo=torch.zeros(P, **i32), hi=torch.zeros(P, **i32))
    s.sptr = _int64s(s.sent.data_ptr() + 4 * n * r for r in range(P))
    s.rptr = torch.zeros(P, dtype=torch.int64, device="cuda")
    s.plan = pkg.A2avPlan(P, 4, s.sptr.data_ptr(), s.sc.data_ptr(), s.sd.data_ptr(), s.rptr.data_ptr(),
                          s.rc.data_ptr(), s.rd.data_ptr())
    return s


def _run_bucket_sort(s):
    pkg, stream = package(), torch.cuda.current_stream().cuda_stream
    pkg.bucket_plan(s.keys.data_ptr(), s.P, s.n, s.key_bits, s.bucket_bits, s.sent.data_ptr(), s.sc.data_ptr(),
                    s.sd.data_ptr(), s.lo.data_ptr(), s.hi.data_ptr(), stream)
    # the ranks' receive buffers lie one after the other, so that one sort orders them all
    total = s.sc.sum(0, dtype=torch.int64)
    torch.add((total.cumsum(0) - total) * 4, s.recv.data_ptr(), out=s.rptr)
    s.plan.execute(stream)
    pkg.local_sort(s.recv.data_ptr(), s.P * s.n, s.key_bits, s.out.data_ptr(), stream)
    return {"sent": s.sent, "send_counts": s.sc, "bucket_lo": s.lo, "bucket_hi": s.hi,
            "recv": s.recv[: s.P * s.n], "sorted": s.out}


def _exact_bucket_sort(case, seed):
    P, n, nb = case["ranks"], case["n"], 1 << case["bucket_bits"]
    keys = _keys(case, seed)
    bucket = (keys >> (case["key_bits"] - case["bucket_bits"])).to(torch.int64)
    rank = torch.arange(P * n, device="cuda") // n
    sent = keys[torch.sort(rank * nb + bucket, stable=True).indices]
    hist = torch.bincount(rank * nb + bucket, minlength=P * nb).reshape(P, nb)
    total, lo, hi, acc, j, prev = hist.sum(0).tolist(), [1] * P, [0] * P, 0, 0, -1
    for b in range(nb):              # rank j takes buckets until the running total reaches (j + 1) n
        acc += total[b]
        if j < P and acc >= (j + 1) * n:
            lo[j], hi[j], prev, j = prev + 1, b, b, j + 1
    before = torch.cat([torch.zeros((P, 1), dtype=torch.int64, device="cuda"), hist.cumsum(1)], 1)
    lo, hi = torch.tensor(lo, device="cuda"), torch.tensor(hi, device="cuda")
    counts = before[:, hi + 1] - before[:, lo]
    counts[:, lo > hi] = 0
    recv = _exchanged(counts.cpu().numpy(), sent.view(torch.uint8), 4).view(torch.int32)
    return {"sent": sent, "send_counts": counts, "bucket_lo": lo, "bucket_hi": hi, "recv": recv,
            "sorted": torch.sort(keys).values}


# ------------------------------------------------------------------ rank programs
def _coll_sizes(case):
    """(elements in, elements out) per rank."""
    return case["count"], case["count"] * (case["ranks"] if case["kind"] == "allgather" else 1)


def _coll_input(case, seed):
    shape, g = (case["ranks"], _coll_sizes(case)[0]), _gen(seed)
    if case["dtype"] == "float64":
        return torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)
    return torch.randint(-(1 << 20), (1 << 20) + 1, shape, dtype=torch.int32, device="cuda", generator=g)


def _prepare_coll(case, seed):
    pkg, P = package(), case["ranks"]
    x = _coll_input(case, seed)
    y = torch.zeros((P, _coll_sizes(case)[1]), dtype=x.dtype, device="cuda")
    seconds = torch.zeros(P, dtype=torch.float64, device="cuda")
    e = x.element_size()
    args = pkg.programs.CollArgs(0, pkg.programs.COLL_KINDS[case["kind"]], pkg.DT[MPI_TYPES[case["dtype"]]], 0, 0,
                                 case["count"], COLL_CALLS, 0, x.data_ptr(), y.data_ptr(), x.shape[1] * e,
                                 y.shape[1] * e, seconds.data_ptr(), 1)
    runtime = pkg.Runtime(P, heap_bytes=64 << 20, timeout_s=20.0)
    return State(x=x, y=y, seconds=seconds, args=args, runtime=runtime)


def _run_coll(s):
    s.runtime.run("coll", s.args)
    return s.y


def _exact_coll(case, seed):
    x, P, kind = _coll_input(case, seed), case["ranks"], case["kind"]
    if kind == "bcast":
        return x[:1].expand(P, -1)
    if kind == "alltoall":
        return x.reshape(P, P, -1).transpose(0, 1).reshape(P, -1)
    if kind == "allgather":
        return x.reshape(1, -1).expand(P, -1)
    total = x.to(torch.float64 if x.dtype.is_floating_point else torch.int64).sum(0)
    if kind == "allreduce":
        return total.expand(P, -1)
    y = torch.zeros((P, x.shape[1]), dtype=total.dtype, device="cuda")
    y[0] = total
    return y


def _prepare_pingpong(case, seed):
    pkg, P, n = package(), case["ranks"], case["bytes"]
    u8 = dict(dtype=torch.uint8, device="cuda")
    s = State(x=torch.zeros((P, n), **u8), y=torch.zeros((P, n), **u8),
              seconds=torch.zeros(P, dtype=torch.float64, device="cuda"),
              wrong=torch.zeros(P, dtype=torch.int64, device="cuda"))
    s.args = pkg.programs.P2pArgs(int(seed), case["mode"], PING_ITERS, 0, 0, n, s.x.data_ptr(), s.y.data_ptr(),
                                  s.seconds.data_ptr(), s.wrong.data_ptr())
    s.runtime = pkg.Runtime(P, heap_bytes=64 << 20, timeout_s=20.0)
    return s


def _run_pingpong(s):
    s.runtime.run("p2p", s.args)
    return {"recv": s.y, "wrong": s.wrong}


# ------------------------------------------------------------------ the cases' five functions
PATHS = {"alltoallv": (_prepare_alltoallv, _run_alltoallv, _exact_alltoallv),
         "reduce": (_prepare_reduce, _run_reduce, _exact_reduce),
         "p2p": (_prepare_p2p, _run_p2p, _exact_p2p),
         "particles": (_prepare_particles, _run_particles, _exact_particles),
         "bucket_sort": (_prepare_bucket_sort, _run_bucket_sort, _exact_bucket_sort),
         "coll": (_prepare_coll, _run_coll, _exact_coll),
         # the payload is drawn by the rank program itself, so there is nothing to compare it with
         "pingpong": (_prepare_pingpong, _run_pingpong, None)}


def prepare(case, seed):
    state = PATHS[case["op"]][0](case, seed)
    state.run = PATHS[case["op"]][1]
    return state


def run(state):
    return state.run(state)


def exact(case, seed):
    f = PATHS[case["op"]][2]
    return f(case, seed) if f else None


def work(case):
    op = case["op"]
    if op == "alltoallv":
        # per step: payload in and out, the four P x P tables
        return {"bytes": case["steps"] * (2 * case["bytes"] + 16 * case["ranks"] ** 2), "flops": 0}
    if op == "reduce":
        n = case["count"] * torch.empty(0, dtype=TORCH_TYPES[case["dtype"]]).element_size()
        return {"bytes": case["ranks"] * n + (case["ranks"] if case["root"] < 0 else 1) * n,
                "flops": (case["ranks"] - 1) * case["count"]}
    if op == "p2p":
        return {"bytes": 2 * case["bytes"] + 24 * case["pairs"], "flops": 0}
    if op == "particles":
        # two steps, each particle's 64 bytes in and out
        return {"bytes": 2 * 128 * case["gx"] * case["gy"] * case["gz"] * case["n0"], "flops": 0}
    if op == "bucket_sort":
        # the keys in; bucketed, exchanged and sorted keys out; count and displacement tables
        return {"bytes": 16 * case["ranks"] * case["n"] + 16 * case["ranks"] ** 2, "flops": 0}
    if op == "coll":
        n_in, n_out = _coll_sizes(case)
        size, P, kind = 4 if case["dtype"] == "int32" else 8, case["ranks"], case["kind"]
        reads = n_in if kind == "bcast" else P * n_in
        writes = n_out if kind == "reduce" else P * n_out
        return {"bytes": COLL_CALLS * size * (reads + writes),
                "flops": COLL_CALLS * (P - 1) * n_in if kind in ("reduce", "allreduce") else 0}
    # every rank sends its message PING_ITERS times, read and written once each
    return {"bytes": 2 * PING_ITERS * case["ranks"] * case["bytes"], "flops": 0}


def tolerance(case):
    """Moved bytes, integers, and folds whose order is part of the contract (rank order): the
    same bits everywhere."""
    return "exact"
