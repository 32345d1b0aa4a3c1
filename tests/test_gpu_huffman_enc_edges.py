"""Huffman encode where a lane's run of symbols meets an edge: streams of
fewer symbols than a lane takes, remainders inside a lane's run and at
partition ends, arrays off their vector alignment, codes that fill a 32-bit
cell exactly, long codes, more partitions than one round of workgroups takes.
Whole bytes: equal to the oracle's stream."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from fzgpumodules_amd import kernels
    return kernels


@pytest.fixture(scope="module")
def orc():
    import oracle
    return oracle


def _encode_at(v, bk4, rev, bklen, off, fine):
    from fzgpumodules_amd._fzh import DeviceBuffer, call, lib, workspace
    eb = v.dtype.itemsize
    d_in = DeviceBuffer(v.nbytes + 32)
    d_in.upload(v, offset=off * eb)
    cap = lib().fzh_huffman_enc_bound(v.size, bklen, eb)
    d_out, d_sz = DeviceBuffer(cap), DeviceBuffer(16)
    d_bk, d_rev = DeviceBuffer.from_array(bk4), DeviceBuffer.from_array(rev)
    ws = workspace(lib().fzh_huffman_enc_ws_bytes(v.size))
    call("fzh_huffman_encode_fine" if fine else "fzh_huffman_encode", None, d_in.ptr + off * eb, v.size, eb, bklen,
         d_bk.ptr, d_rev.ptr, d_out.ptr, cap, d_sz.ptr, ws.ptr, ws.nbytes)
    return d_out.download(np.uint8, int(d_sz.download(np.uint64, 1)[0]))


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32])
@pytest.mark.parametrize("fine", [False, True])
def test_remainders_and_alignment(gpu, orc, dtype, fine):
    rng = np.random.default_rng(3)
    f = np.zeros(256, np.uint32)
    f[:200] = rng.integers(900, 1000, 200)  # codes of 7 and 8 bits
    bk4, rev = orc.huffman_book(f, np.dtype(dtype).itemsize)
    sl = 1024 if fine else 768
    for n in (1, 11, 13, 64, sl - 1, sl, sl + 1, sl + sl // 64 - 1, 4 * sl, 5 * sl + 7):
        v = rng.integers(0, 200, n).astype(dtype)
        from test_cpu_oracle import huffman_stream_def
        want = huffman_stream_def(v, bk4, rev, 256, sl)
        for off in (0, 1):
            assert np.array_equal(_encode_at(v, bk4, rev, 256, off, fine), want), (n, off)


@pytest.mark.parametrize("kind", ["eight_bits", "one_bit", "to_26_bits"])
def test_cells(gpu, orc, kind):
    """Codes whose runs end on cell boundaries, share a cell among many
    lanes, or span cells."""
    from test_cpu_oracle import huffman_stream_def
    rng = np.random.default_rng(8)
    if kind == "eight_bits":
        f, pick = np.full(256, 10, np.uint32), lambda n: rng.integers(0, 256, n)
    elif kind == "one_bit":
        f, pick = np.array([1000, 1, 1, 0], np.uint32), lambda n: (rng.random(n) < 0.01).astype(int)
    else:
        f = np.maximum(2.0 ** (27 - 0.5 * np.arange(1024)), 20).astype(np.uint32)
        pick = lambda n: rng.integers(0, 1024, n)  # noqa: E731
    bk4, rev = orc.huffman_book(f, 2)
    assert (bk4[f > 0] >> 27).max() <= 26
    v = pick(768 * 9 + 500).astype(np.uint16)
    assert np.array_equal(_encode_at(v, bk4, rev, f.size, 0, False), huffman_stream_def(v, bk4, rev, f.size, 768))


def test_many_partitions(gpu, orc):
    v = np.minimum(np.abs(np.random.default_rng(1).laplace(0, 6, 768 * 4 * 4096 * 2 + 777)), 255).astype(np.uint8)
    assert np.array_equal(gpu.huffman_encode(v, 256), orc.huffman_encode(v, 256))
