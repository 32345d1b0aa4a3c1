"""Huffman decode of long streams (one lane per partition) on streams made
by repeating a block of partitions that the numpy stream definition wrote:
every level of the decode tables and the codes past them, partition lengths
that segments of 16 symbols divide and do not, remainders of the last
partition, constant partitions, and corrupt partition metadata.  The result
is compared with the repeated symbols themselves (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LONG = 32768 * 768  # symbols from which the decoder gives every partition a lane


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
    assert n >= LONG
    got = gpu.huffman_decode(s, dtype, n)
    want = np.concatenate([np.tile(block, reps), tail])
    assert np.array_equal(got, want)


@pytest.mark.parametrize("what", ["bits", "entry"])
@pytest.mark.parametrize("part", [0, 20000, -1])
def test_long_stream_rejects_corrupt_partition(gpu, orc, what, part):
    bk4, rev, bklen, f = _book(orc, "gauss", 2)
    rng = np.random.default_rng(9)
    block = rng.choice(bklen, 128 * 768, p=f).astype(np.uint16)
    s, n = _repeat(block, block[:100], bk4, rev, bklen, 768, LONG // block.size)
    e = s[40:64].view(np.uint32)
    nb, en = s[e[2]:e[3]].view(np.uint32), s[e[3]:e[4]].view(np.uint32)
    if what == "bits":
        nb[part] += 1 if nb[part] % 32 else -1
    else:
        en[part] = (e[5] - e[4]) // 4
    with pytest.raises(ValueError):
        gpu.huffman_decode(s, np.uint16, n)
