"""The verify kernel's lane arithmetic (csrc/verify_kernel.cuh), restated on the
CPU: `reduce_rows` over the 16 (or 8) blocks of a 4x4x1 matrix instruction, the
loads' cover of a block of rows, `udiv`, and the runs of 16-bit elements that start in
either half of a dword (`load_run`)."""

import random

import pytest


def _swap32(x, y):
    return x[:32] + y[:32], x[32:] + y[32:]


def _swap16(x, y):
    rows = lambda a: [a[16 * i:16 * i + 16] for i in range(4)]  # noqa: E731
    a, b = rows(x), rows(y)
    return a[0] + b[0] + a[2] + b[2], a[1] + b[1] + a[3] + b[3]


def _add(p):
    return [a + b for a, b in zip(*p)]


def _ror(x, n):
    return [x[16 * (i // 16) + (i % 16 - n) % 16] for i in range(64)]


def test_reduce_rows_sums_the_blocks():
    rng = random.Random(1)
    acc = [[rng.randrange(1 << 20) for _ in range(64)] for _ in range(4)]  # register r, lane 4*block + column
    x = _add(_swap16(_add(_swap32(acc[0], acc[2])), _add(_swap32(acc[1], acc[3]))))
    x = _add((x, _ror(x, 8)))
    x = _add((x, _ror(x, 4)))
    for lane in range(64):
        r, col = lane >> 4, lane & 3
        assert x[lane] == sum(acc[r][4 * kb + col] for kb in range(16))


def test_reduce_rows8_sums_the_blocks_of_each_half():
    """Rows over 8 blocks: lo holds rows 0 (even 16 lanes) and 1 (odd) of each half's
    tile, hi rows 2 and 3."""
    rng = random.Random(3)
    acc = [[rng.randrange(1 << 20) for _ in range(64)] for _ in range(4)]
    for first in (0, 2):
        x = _add(_swap16(acc[first], acc[first + 1]))
        x = _add((x, _ror(x, 8)))
        x = _add((x, _ror(x, 4)))
        for lane in range(64):
            half, r, col = lane >> 5, first + ((lane >> 4) & 1), lane & 3
            assert x[lane] == sum(acc[r][32 * half + 4 * kb + col] for kb in range(8))


def test_result_rows_over_8_blocks():
    """Copies 2g and 2g + 1 keep lo and hi of load g: lane and register give row
    8*(bq >> 1) + 4*(lane >> 5) + 2*(bq & 1) + (lane >> 4 & 1), every row once per column."""
    got = {}
    for lane in range(64):
        bq = (lane >> 2) & 3
        g, hi, half = bq >> 1, bq & 1, lane >> 5
        source = 8 * g + 4 * half + 2 * hi + ((lane >> 4) & 1)  # load g's rows 8g + 4*half + (0..3)
        row = 8 * (bq >> 1) + 4 * (lane >> 5) + 2 * (bq & 1) + ((lane >> 4) & 1)
        assert row == source and (row, lane & 3) not in got
        got[row, lane & 3] = lane
    assert len(got) == 64


@pytest.mark.parametrize("N", [16, 8])
def test_gram_lanes(N):
    """gram_lane(s, c) names a lane that holds row s % 4, column c % 4 of the result."""
    for s in range(8):
        for c in range(16):
            lane = (16 * (s & 3) if N == 16 else 16 * (s & 1) + 4 * ((s >> 1) & 1)) + (c & 3)
            row = lane >> 4 if N == 16 else ((lane >> 4) & 1) + 2 * ((lane >> 2) & 1)
            assert row == s % 4 and (lane & 3) == c % 4


@pytest.mark.parametrize("N,J", [(16, 1), (16, 2), (16, 4), (8, 1)])
@pytest.mark.parametrize("block", [16, 8])
def test_block_loads_are_whole_row_runs(N, J, block):
    """Register g*J + j of a lane holds chunk N*j + kb of row ROWS*g + lr: each chunk
    once, every load 64 / N runs of N consecutive chunks."""
    rows = 64 // N
    if block % rows:
        pytest.skip("not a block of this split")
    seen = []
    for g in range(block // rows):
        for j in range(J):
            at = []
            for lane in range(64):
                kb, ij = (lane >> 2) & (N - 1), lane & 3
                lr = ij if N == 16 else 4 * (lane >> 5) + ij
                at.append((rows * g + lr, N * j + kb))
            assert sorted(at) == [(rows * g + r, N * j + c) for r in range(rows) for c in range(N)]
            seen += at
    assert sorted(seen) == [(r, c) for r in range(block) for c in range(N * J)]


def test_udiv_is_exact():
    rng = random.Random(2)
    ds = [1, 2, 3, 5, 7, 12, 31, 64, 1000, 65535, 65537, (1 << 31) - 1, 1 << 31, (1 << 32) - 1]
    ds += [rng.randrange(1, 1 << rng.randrange(1, 33)) for _ in range(300)]
    for d in ds:
        m = 0xFFFFFFFF // d
        xs = {0, 1, d - 1, d, d + 1, 2 * d - 1, 2 * d, 0x7FFFFFFF, 0xFFFFFFFF, (0xFFFFFFFF // d) * d, (0xFFFFFFFF // d) * d - 1}
        xs |= {rng.randrange(1 << 32) for _ in range(50)}
        for x in xs:
            if not 0 <= x < 1 << 32:
                continue
            q = (x * m) >> 32
            q += x - q * d >= d
            assert q == x // d, (x, d)


@pytest.mark.parametrize("N", [4, 8])
@pytest.mark.parametrize("first", range(8))
def test_runs_of_16_bit_elements(N, first):
    """A run from any element: the dwords read hold elements of the run only,
    and the funnel shift lines them up."""
    elems = [0x1000 + i for i in range(32)]
    words = [elems[2 * i] | elems[2 * i + 1] << 16 for i in range(16)]
    off = first * 2
    odd = off & 2
    at = off // 4
    got = words[at:at + N // 2] + [words[at + N // 2] if odd else 0]
    touched = range(at, at + N // 2 + (1 if odd else 0))
    assert all(2 * w + 1 >= first and 2 * w < first + N for w in touched)
    sh = 16 if odd else 0
    out = []
    for i in range(N // 2):
        u = (((got[i + 1] << 32) | got[i]) >> sh) & 0xFFFFFFFF
        out += [u & 0xFFFF, u >> 16]
    assert out == elems[first:first + N]


@pytest.mark.parametrize("chunks", [16, 8])
def test_both_forms_sum_the_chunks_in_one_order(chunks):
    """The tree of reduce_rows / reduce_rows8 over a row's chunks (kb ^ 8, ^ 4, ^ 2, ^ 1
    by lane) and of sum_results (chunk 4j + block: j, then block ^ 2, ^ 1) add the
    same pairs at every level, so the two give the same bits."""
    def pair(level, bit):
        return {c: frozenset((level[c], level[c ^ bit])) for c in level}

    lanes = {c: c for c in range(chunks)}
    for bit in ([8] if chunks == 16 else []) + [4, 2, 1]:
        lanes = pair(lanes, bit)

    def product(j):
        return {b: 4 * j + b for b in range(4)}

    def add(x, y):
        return {b: frozenset((x[b], y[b])) for b in x}

    if chunks == 16:
        x = add(add(product(0), product(2)), add(product(1), product(3)))
    else:
        x = add(product(0), product(1))
    got = frozenset((frozenset((x[0], x[2])), frozenset((x[1], x[3]))))
    assert all(v == got for v in lanes.values())
