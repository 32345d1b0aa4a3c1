"""Bit packing, the code maximum and the segment gather at the
edges of their vector paths: fewer elements than one 16-element group,
remainders, arrays off 16-byte alignment, every width of every element type.
All results are whole bytes: equal to the oracle's or to numpy's."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fzh():
    from fzgpumodules_amd import _fzh
    return _fzh


@pytest.fixture(scope="module")
def orc():
    import oracle
    return oracle


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 4096, 70_003])
@pytest.mark.parametrize("shift", [0, 1])
def test_bitpack_every_width(fzh, orc, dtype, n, shift):
    es = np.dtype(dtype).itemsize
    rng = np.random.default_rng(n + es)
    for nbits in (1, 2, 4, 8, 16, 32):
        if nbits > 8 * es:
            continue
        v = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(dtype)  # high bits too: the packing masks them
        nout = (n * nbits + 7) // 8
        d_in, d_out = fzh.DeviceBuffer(es * (n + 1) + 16), fzh.DeviceBuffer.zeros(nout + 32)
        d_in.upload(v, offset=shift * es)
        fzh.call("fzh_bitpack_enc", None, d_in.ptr + shift * es, n, es, nbits, d_out.ptr)
        got = d_out.download(np.uint8, nout + 16)
        want = orc.bitpack_enc(v & dtype((1 << nbits) - 1), nbits)
        assert np.array_equal(got[:nout], want) and not got[nout:].any()
        d_back = fzh.DeviceBuffer.zeros(es * (n + 1) + 16)
        fzh.call("fzh_bitpack_dec", None, d_out.ptr, n, es, nbits, d_back.ptr + shift * es)
        back = d_back.download(dtype, n + 1)
        assert np.array_equal(back[shift:shift + n], v & dtype((1 << nbits) - 1))


@pytest.mark.parametrize("n", [1, 7, 8, 4099, 2_000_003])
@pytest.mark.parametrize("where", [0, -1, "middle"])
def test_max_finds_one_peak(fzh, n, where):
    v = np.zeros(n, np.uint16)
    v[n // 2 if where == "middle" else where] = 60001
    ws = fzh.workspace(fzh.lib().fzh_max_u32_ws_bytes())
    m = fzh.DeviceBuffer(16)
    for off in (0, 2):
        d = fzh.DeviceBuffer(v.nbytes + 16)
        d.upload(v, offset=off)
        fzh.call("fzh_max_u32", None, d.ptr + off, n, 2, m.ptr, ws.ptr, ws.nbytes)
        assert int(m.download(np.uint32, 1)[0]) == 60001


@pytest.mark.parametrize("n_segs", [1, 3, 60, 5000])
def test_gather_segments(fzh, n_segs):
    """Empty, short, long and unaligned segments; bytes between them stay."""
    rng = np.random.default_rng(n_segs)
    sizes = rng.integers(0, 300 if n_segs > 100 else 70_000, n_segs)
    sizes[0] = 0 if n_segs > 1 else 1_000_001
    src_off = np.r_[0, np.cumsum(sizes + rng.integers(0, 20, n_segs))].astype(np.int64)
    dst_off = np.r_[0, np.cumsum(sizes + rng.integers(1, 20, n_segs))].astype(np.int64)
    if n_segs % 2 == 0:  # aligned ends
        src_off = np.r_[0, np.cumsum((sizes + 15) // 16 * 16)].astype(np.int64)
        dst_off = np.r_[0, np.cumsum((sizes + 31) // 16 * 16)].astype(np.int64)
    data = rng.integers(0, 256, int(src_off[-1]) + 16).astype(np.uint8)
    want = np.full(int(dst_off[-1]) + 16, 7, np.uint8)
    d_src, d_dst = fzh.DeviceBuffer.from_array(data), fzh.DeviceBuffer.from_array(want)
    desc = np.zeros(n_segs, np.dtype([("s", np.uint64), ("d", np.uint64), ("n", np.uint64)]))
    for i, n in enumerate(sizes):
        desc[i] = (d_src.ptr + src_off[i], d_dst.ptr + dst_off[i], n)
        want[dst_off[i]:dst_off[i] + n] = data[src_off[i]:src_off[i] + n]
    d_desc = fzh.DeviceBuffer.from_array(desc)
    fzh.call("fzh_gather", None, d_desc.ptr, n_segs)
    assert np.array_equal(d_dst.download(np.uint8, want.size), want)


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32])
@pytest.mark.parametrize("n", [8191, 8192, 8193, 16_384, 16_385, 32_768, 32_769])  # one workgroup, then partial maxima
@pytest.mark.parametrize("at", [0, 8190, -1])
def test_max_around_one_workgroup(fzh, dtype, n, at):
    v = np.full(n, 3, dtype)
    v[at] = 201
    ws = fzh.workspace(fzh.lib().fzh_max_u32_ws_bytes())
    m = fzh.DeviceBuffer(16)
    d = fzh.DeviceBuffer.from_array(v)
    fzh.call("fzh_max_u32", None, d.ptr, n, v.itemsize, m.ptr, ws.ptr, ws.nbytes)
    assert int(m.download(np.uint32, 1)[0]) == 201


@pytest.mark.parametrize("nbytes", [1, 15, 16, 255, 256, 257, 272])  # a byte a thread up to 256
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n_segs", [2, 5000])
def test_gather_of_small_segments(fzh, nbytes, shift, n_segs):
    step = 288
    data = np.random.default_rng(nbytes).integers(0, 256, n_segs * step + 16).astype(np.uint8)
    d_src, d_dst = fzh.DeviceBuffer.from_array(data), fzh.DeviceBuffer.from_array(np.full(n_segs * step, 7, np.uint8))
    desc = np.zeros(n_segs, np.dtype([("s", np.uint64), ("d", np.uint64), ("n", np.uint64)]))
    at = np.arange(n_segs, dtype=np.uint64) * step
    desc["s"], desc["d"], desc["n"] = d_src.ptr + shift + at, d_dst.ptr + at, nbytes
    d_desc = fzh.DeviceBuffer.from_array(desc)
    fzh.call("fzh_gather", None, d_desc.ptr, n_segs)
    got = d_dst.download(np.uint8, n_segs * step).reshape(n_segs, step)
    assert np.array_equal(got[:, :nbytes], data[shift:shift + n_segs * step].reshape(n_segs, step)[:, :nbytes])
    assert (got[:, nbytes:] == 7).all()
