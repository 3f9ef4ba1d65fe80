"""The short rows' copy (runtime/batched.h: a2av_copy_short, a2av_assemble_line, a2av_row_end) on the
CPU.  test_kernel_code runs the kernels' own code over random layouts, whole-row windows of up
to 64 ranks and the long rows' ends among them.  test_short_row_lines is a model of the design
alone: the window of segments found by a search (as with more than 64 ranks), the lane's
bisection, the two-segment funnel and the piecewise assembly are restated and every row byte
must be written once, reading no byte outside its segment."""
import numpy as np
import pytest

from host_build import run_check

WINDOW = 512


def test_kernel_code(tmp_path):
    run_check("a2av_short_check", tmp_path, sanitize=True)


def assemble(rbase, rbytes, line, at, read):
    """{row byte: value} of a2av_assemble_line; read(a, n) is a load of n bytes."""
    off = line * 16 - rbase
    b0 = 0 if off >= 0 else 16 if off <= -16 else -off
    b1 = 16 if rbytes - off >= 16 else rbytes - off
    got, pos = {}, b0
    while pos < b1:
        st, en, D = at(off + pos)
        end, start = en - off, st - off
        e = min(end, b1)
        src = line * 16 + D
        if end - start >= 16:
            f = min(max(start, 0), end - 16)
            assert -15 <= f <= 15
            x = read(src + f, 16)
            y = [x[i - f] if 0 <= i - f < 16 else 0 for i in range(16)]
        else:
            n = e - pos
            assert 0 < n < 16
            y = [0] * pos + read(src + pos, n) + [0] * (16 - pos - n)
        for i in range(pos, e):
            got[off + i] = y[i]
        pos = e
    return got


@pytest.mark.parametrize("seed", range(12))
@pytest.mark.parametrize("P,mean,phase", [(1, 5, 3), (3, 700, 9), (16, 40, 0), (40, 17, 15), (700, 3, 1), (1300, 2, 6),
                                          (64, 1, 8)])
def test_short_row_lines(P, mean, phase, seed):
    rng = np.random.default_rng(seed * 1000 + P)
    size = rng.poisson(mean, P)
    size[rng.random(P) < 0.3] = 0
    if P > 600 and seed % 2:
        size[20:20 + WINDOW + 30] = 0          # more empty segments in one line than a window holds
    end = np.cumsum(size)
    rbytes = int(end[-1])
    if rbytes == 0:
        return
    rbase = 4096 + phase
    gap = np.cumsum(size + rng.integers(0, 9, P)) + 100000
    src = gap - size                            # each segment's bytes, apart from the others'
    memory = {}
    for s in range(P):
        for i in range(size[s]):
            memory[int(src[s]) + i] = int(rng.integers(0, 256))
    want = [memory[int(src[s]) + i] for s in range(P) for i in range(size[s])]

    def read(a, n):
        return [memory[a + i] for i in range(n)]        # KeyError: outside every segment

    def seg(q):
        k = int(np.searchsorted(end, q, side="right"))
        st = int(end[k - 1]) if k else 0
        return st, int(end[k]), int(src[k]) - (rbase + st)

    written = {}

    def write(q, v):
        assert 0 <= q < rbytes and q not in written
        written[q] = v

    lend = (rbase + rbytes + 15) >> 4
    for line0 in range((rbase >> 7) << 3, lend, 64):
        line1 = min(line0 + 64, lend)
        pos = line0
        most = min(WINDOW, 2 * 16 * (line1 - pos) * P // rbytes + 16)
        while pos < line1:
            o = max(pos * 16 - rbase, 0)
            s0 = int(np.searchsorted(end, o, side="right"))
            n = min(P - s0, most)
            E = [int(end[s0 + k]) - o for k in range(n)]
            first = (int(end[s0 - 1]) if s0 else 0) - o
            pend = line1 if s0 + n >= P else (rbase + E[-1] + o) >> 4
            pend = min(pend, line1)
            if pend <= pos:
                for q, v in assemble(rbase, rbytes, pos, seg, read).items():
                    write(q, v)
                pos += 1
                continue

            def at(q):
                k = next(i for i in range(n) if E[i] > q - o or i == n - 1)
                assert E[k] > q - o
                st = o + (E[k - 1] if k else first)
                return st, o + E[k], int(src[s0 + k]) - (rbase + (int(end[s0 + k - 1]) if s0 + k else 0))

            for line in range(pos, pend):
                off = line * 16 - rbase
                if off <= -16:
                    continue
                q = max(off, 0) - o
                k = 0
                b = 1 << ((n - 1).bit_length() - 1) if n > 1 else 0
                while b:
                    if k + b <= n - 1 and E[k + b - 1] <= q:
                        k += b
                    b >>= 1
                if not (off < 0 or off + 16 > rbytes):
                    e = E[k]
                    D = int(src[s0 + k]) - (rbase + (int(end[s0 + k - 1]) if s0 + k else 0))
                    if e - q >= 16:
                        for i, v in enumerate(read(line * 16 + D, 16)):
                            write(off + i, v)
                        continue
                    k2 = k + 1
                    while k2 < n - 1 and E[k2] <= e:
                        k2 += 1
                    st = E[k - 1] if k else first
                    if k2 < n and E[k2] - e >= 16 and e - st >= 16:
                        a = e - q
                        D2 = int(src[s0 + k2]) - (rbase + int(end[s0 + k2 - 1]))
                        both = read(line * 16 + a - 16 + D, 16) + read(line * 16 + a + D2, 16)
                        for i in range(16):
                            write(off + i, both[16 - a + i])
                        continue
                for x, v in assemble(rbase, rbytes, line, at, read).items():
                    write(x, v)
            pos = pend
    assert [written[q] for q in range(rbytes)] == want
