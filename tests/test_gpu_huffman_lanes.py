"""Huffman decode of long streams (one lane or one wave per partition, as the
stream says) on streams made by repeating a block of partitions that the numpy
stream definition wrote: every level of the decode tables and the codes past
them, partition lengths that segments of 16 symbols divide and do not, remainders
of the last partition, constant partitions, streams on both sides of the choice,
and corrupt partition metadata.  The result is compared with the repeated symbols
themselves (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LONG = 65536 * 768  # symbols from which every stream of the cases but two is decoded by lanes
MIN = 32768 * 768   # symbols from which any is


def by_lanes(s, n, itemsize):
    """The decoder's choice by its costs (dec_by_lanes; runs are not looked for)."""
    sublen, parts = s[4:12].view(np.uint32).tolist()
    e = s[40:64].view(np.uint32)
    if n < MIN or sublen % 16 or sublen > 1024 or s[e[1]:e[2]].view(np.uint32)[33] == 1:
        return False
    bits = 8 * float(e[5] - e[4]) / n
    wave = 1.35 + (0.35 if itemsize == 1 else 0.4) * bits + 0.06 * max(0.0, 32 / bits - sublen / 64)
    return bool(wave * parts > (156 if itemsize == 1 else 168) * sublen)


@pytest.fixture(scope="module")
def gpu():
    from fzgpumodules_amd import kernels
    return kernels


@pytest.fixture(scope="module")
def orc():
    import oracle
    return oracle


def _book(orc, book, itemsize):
    """(codebook, revbook, bklen, frequency-free symbol draw)"""
    bklen = 256 if itemsize == 1 else 1024
    i = np.arange(bklen)
    if book == "gauss":
        f = np.exp(-0.5 * ((i - bklen // 2) / (bklen / 30)) ** 2)
    elif book == "narrow":
        f = np.exp(-np.abs(i - bklen // 2) / 1.2)
    elif book == "tail":  # every length from 1 to past the tables' levels
        f = 2.0 ** (-0.09 * i - 0.5 * np.minimum(i, 6))
    else:  # one symbol
        f = np.where(i == 7, 1000.0, 0.0)
    if book != "one":
        f = np.maximum(f / f.sum(), 3e-8)  # codes of at most 26 bits
    f = f / f.sum()
    bk4, rev = orc.huffman_book(np.maximum(f * 1e9, f > 0).astype(np.uint32), itemsize)
    return bk4, rev, bklen, f


def _repeat(block, tail, bk4, rev, bklen, sublen, reps):
    """The stream of `block` (whole partitions) `reps` times, then `tail`."""
    from test_cpu_oracle import huffman_stream_def

    def parts(v):
        s = huffman_stream_def(v, bk4, rev, bklen, sublen)
        e = s[40:64].view(np.uint32)
        return s[e[2]:e[3]].view(np.uint32), s[e[4]:e[5]].view(np.uint32), s

    nb, ce, s0 = parts(block)
    nbit, cells = np.tile(nb, reps), np.tile(ce, reps)
    if tail.size:
        tn, tc, _ = parts(tail)
        nbit, cells = np.r_[nbit, tn], np.r_[cells, tc]
    ncell = (nbit.astype(np.int64) + 31) // 32
    entry = np.r_[0, np.cumsum(ncell)[:-1]].astype(np.uint32)
    h = s0[:128].copy()
    n = block.size * reps + tail.size
    h[4:12] = np.array([sublen, nbit.size], np.int32).view(np.uint8)
    h[16:40] = np.array([n, nbit.sum(dtype=np.uint64), cells.size], np.uint64).view(np.uint8)
    e = np.cumsum([0, 128, rev.size, 4 * nbit.size, 4 * nbit.size, 4 * cells.size]).astype(np.uint32)
    h[40:64] = e.view(np.uint8)
    return np.concatenate([h, rev, nbit.view(np.uint8), entry.view(np.uint8), cells.view(np.uint8)]), n


CASES = [  # book, type, partition length, symbols beyond LONG, tail symbols of the block's kind
    ("gauss", np.uint16, 768, 0), ("gauss", np.uint16, 768, 769), ("gauss", np.uint8, 768, 5),
    ("tail", np.uint16, 768, 100), ("tail", np.uint8, 768, 31), ("tail", np.uint16, 1024, 1000),
    ("gauss", np.uint16, 48, 47), ("gauss", np.uint16, 333, 1), ("one", np.uint16, 768, 3),
]


@pytest.mark.parametrize("book,dtype,sublen,extra", CASES)
def test_long_streams(gpu, orc, book, dtype, sublen, extra):
    bk4, rev, bklen, f = _book(orc, book, np.dtype(dtype).itemsize)
    rng = np.random.default_rng(sublen + extra)
    if book == "one":
        sym = np.full(97 * sublen, 7)
    else:
        # partitions of typical symbols, of any symbol alike, and of the rarest
        typical = rng.choice(bklen, 64 * sublen, p=f)
        sym = np.concatenate([typical, rng.integers(0, bklen, 32 * sublen), rng.integers(bklen - 40, bklen, sublen)])
    block = sym.astype(dtype)
    if book == "tail" and dtype == np.uint16:  # codes of more bits than the first table's and its chain's
        lens = bk4[block.astype(np.int64)] >> 27
        assert lens.min() <= 3 and lens.max() >= 25
    reps = -(-LONG // block.size)
    tail = block[:extra] if extra <= block.size else block
    s, n = _repeat(block, tail, bk4, rev, bklen, sublen, reps)
    assert n >= LONG and by_lanes(s, n, block.itemsize) == (book != "one" and sublen != 333)
    got = gpu.huffman_decode(s, dtype, n)
    want = np.concatenate([np.tile(block, reps), tail])
    assert np.array_equal(got, want)


@pytest.mark.parametrize("what", ["bits", "entry"])
@pytest.mark.parametrize("part", [0, 20000, -1])  # (lanes and waves)
@pytest.mark.parametrize("size", [LONG, MIN])
def test_long_stream_rejects_corrupt_partition(gpu, orc, what, part, size):
    bk4, rev, bklen, f = _book(orc, "gauss" if size == LONG else "narrow", 2)
    rng = np.random.default_rng(9)
    block = rng.choice(bklen, 128 * 768, p=f).astype(np.uint16)
    s, n = _repeat(block, block[:100], bk4, rev, bklen, 768, -(-size // block.size))
    assert by_lanes(s, n, 2) == (size == LONG)
    e = s[40:64].view(np.uint32)
    nb, en = s[e[2]:e[3]].view(np.uint32), s[e[3]:e[4]].view(np.uint32)
    if what == "bits":
        nb[part] += 1 if nb[part] % 32 else -1
    else:
        en[part] = (e[5] - e[4]) // 4
    with pytest.raises(ValueError):
        gpu.huffman_decode(s, np.uint16, n)


# streams around the choice, which the encoder writes or a program could
CHOICES = [("narrow", np.uint16, 768, MIN, False), ("narrow", np.uint16, 768, LONG, True),
           ("narrow", np.uint8, 768, MIN, False), ("narrow", np.uint8, 1024, LONG, False),
           ("gauss", np.uint16, 1024, MIN, False), ("gauss", np.uint16, 1024, LONG, True),
           ("gauss", np.uint16, 2000, LONG, False), ("gauss", np.uint8, 4096, MIN, False),
           ("gauss", np.uint16, 65536, MIN, False), ("narrow", np.uint8, 1 << 20, MIN, False),
           ("one", np.uint8, 768, MIN, False), ("one", np.uint16, 1024, LONG, False)]


@pytest.mark.parametrize("book,dtype,sublen,size,lanes", CHOICES)
def test_choice(gpu, orc, book, dtype, sublen, size, lanes):
    bk4, rev, bklen, f = _book(orc, book, np.dtype(dtype).itemsize)
    rng = np.random.default_rng(sublen)
    k = max(1, 98304 // sublen) * sublen
    block = (np.full(k, 7) if book == "one" else rng.choice(bklen, k, p=f)).astype(dtype)
    reps = -(-size // block.size)
    tail = block[:min(sublen, 777)]
    s, n = _repeat(block, tail, bk4, rev, bklen, sublen, reps)
    assert n >= MIN and by_lanes(s, n, block.itemsize) == lanes
    assert np.array_equal(gpu.huffman_decode(s, dtype, n), np.concatenate([np.tile(block, reps), tail]))


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16])
@pytest.mark.parametrize("share", [0.1, 0.9])
def test_runs(gpu, orc, dtype, share):
    """Partitions of one repeated code (lanes take streams of enough of them) among others."""
    bk4, rev, bklen, f = _book(orc, "narrow", np.dtype(dtype).itemsize)
    rng = np.random.default_rng(7)
    block = rng.choice(bklen, 128 * 768, p=f).astype(dtype)
    code = int(np.argsort(-f)[4])  # a few bits
    for p in rng.permutation(128)[:int(128 * share)]:
        block[768 * p:768 * (p + 1)] = code
    reps = -(-MIN // block.size)
    s, n = _repeat(block, block[:5], bk4, rev, bklen, 768, reps)
    assert not by_lanes(s, n, block.itemsize)
    assert np.array_equal(gpu.huffman_decode(s, dtype, n), np.concatenate([np.tile(block, reps), block[:5]]))


@pytest.mark.parametrize("book,sublen,us", [("gauss", 333, 800), ("gauss", 65536, 3500)])
def test_time_of_other_partition_lengths(orc, book, sublen, us):
    """Lengths that lanes don't take: a wave per partition (240 and 1180 us; 2660 and
    8160 where a wave took 64 partitions in turn, or a lane one of these)."""
    from fzgpumodules_amd._fzh import DeviceBuffer, Event, call, synchronize
    bk4, rev, bklen, f = _book(orc, book, 2)
    k = max(1, 98304 // sublen) * sublen
    block = np.random.default_rng(3).choice(bklen, k, p=f).astype(np.uint16)
    s, n = _repeat(block, block[:5], bk4, rev, bklen, sublen, -(-MIN // block.size))
    d, y, st = DeviceBuffer.from_array(s), DeviceBuffer(2 * n), DeviceBuffer.zeros(16)
    best = 1e9
    for _ in range(6):
        a, b = Event(), Event()
        a.record()
        call("fzh_huffman_decode", None, d.ptr, s.size, 2, y.ptr, n, st.ptr)
        b.record()
        synchronize()
        best = min(best, 1e3 * a.elapsed_ms(b))
    assert st.download(np.int32, 1)[0] == 0
    assert best < us
