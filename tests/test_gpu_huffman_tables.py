"""The decode tables' levels behind the first, at entry counts around a wave:
books with dyadic frequencies, so their code lengths are known.  `c` of the
first table's 2048 entries are prefixes of codes of 11 + d bits, which makes the
second level's c << d entries; `deep` hangs a chain of codes up to 25 bits under
one of them, for the levels after it.  Every symbol occurs; the decoded symbols
are the stream's (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(1, 1, False), (3, 1, False), (5, 3, True), (1, 6, True), (31, 1, False), (33, 1, True), (16, 2, False),
         (17, 2, True), (63, 1, False), (65, 1, True), (100, 3, False), (129, 2, True)]


def _frequencies(c, d, deep, bklen):
    """One symbol per code; frequency 2^(25 - length)."""
    lens, left = [11 + d] * (c << d), 2048 - c
    for bit in range(11):  # the other prefixes, as few codes as possible
        if left >> bit & 1:
            lens.append(11 - bit)
    if deep:
        first = lens.pop(0)
        lens += list(range(first + 1, 26)) + [25]
    f = np.zeros(bklen, np.uint32)
    at = np.random.default_rng(c * 64 + d).permutation(bklen)[:len(lens)]
    f[at] = 1 << (25 - np.array(lens))
    return f, at, np.array(lens)


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32])
@pytest.mark.parametrize("c,d,deep", CASES)
def test_short_streams(gpu, orc, c, d, deep, dtype):
    from test_cpu_oracle import huffman_stream_def
    bklen = 256 if dtype == np.uint8 else 1024
    if (c << d) + 30 > bklen:
        c = (bklen - 30) >> d
    f, sym, lens = _frequencies(c, d, deep, bklen)
    bk4, rev = orc.huffman_book(f, np.dtype(dtype).itemsize)
    assert np.array_equal(bk4[sym] >> 27, lens)
    v = np.random.default_rng(c).choice(sym, 9 * 768 + 13).astype(dtype)
    v[:sym.size] = sym
    s = huffman_stream_def(v, bk4, rev, bklen, 768)
    assert np.array_equal(gpu.huffman_decode(s, dtype, v.size), v)


@pytest.mark.parametrize("c,d,deep", [(17, 2, True), (33, 1, False)])
def test_long_streams(gpu, orc, c, d, deep):
    from test_gpu_huffman_lanes import LONG, _repeat
    f, sym, _ = _frequencies(c, d, deep, 1024)
    bk4, rev = orc.huffman_book(f, 2)
    block = np.random.default_rng(d).choice(sym, 64 * 768).astype(np.uint16)
    block[:sym.size] = sym
    reps = -(-LONG // block.size)
    s, n = _repeat(block, block[:100], bk4, rev, 1024, 768, reps)
    assert np.array_equal(gpu.huffman_decode(s, np.uint16, n), np.concatenate([np.tile(block, reps), block[:100]]))


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32])
@pytest.mark.parametrize("sublen", [768, 333, 5])
@pytest.mark.parametrize("n", [1, 15, 767, 769, 100_003])
def test_constant(gpu, orc, dtype, sublen, n):
    """One symbol, whose code has no bits: partitions on and off 16-byte alignment."""
    from test_cpu_oracle import huffman_stream_def
    bklen = 256 if dtype == np.uint8 else 1024
    f = np.zeros(bklen, np.uint32)
    f[201] = n
    bk4, rev = orc.huffman_book(f, np.dtype(dtype).itemsize)
    v = np.full(n, 201, dtype)
    assert np.array_equal(gpu.huffman_decode(huffman_stream_def(v, bk4, rev, bklen, sublen), dtype, n), v)
