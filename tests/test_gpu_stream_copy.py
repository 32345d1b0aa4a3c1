"""Coders that store their stream in the caller's buffer as well as in the
pool's: RLE and Huffman of each code size behind a quantizer or the predictor,
sizes around their tiles and partitions, books longer than the stream, the fine
layout, and an input that lies in the output buffer (which takes the copy),
byte for byte the pool-owned call's result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fzh():
    from fzgpumodules_amd import _fzh
    return _fzh


def _pipe(n, coder, cb):
    from fzgpumodules_amd.pipeline import Pipeline
    p = Pipeline(4 * n)
    radius = 100 if cb == 1 else 512
    if cb == 4:
        a = p.add_quantizer(1e-2, mode="ABS", quant_radius=radius, outlier_capacity=0.3, zigzag=True, code_bytes=4)
    else:
        a = p.add_lorenzo(1e-2, quant_radius=radius, outlier_capacity=0.3, zigzag=True, code_bytes=cb)
    b = p.add_rle(cb) if coder == "rle" else p.add_huffman(cb, 256 if cb == 1 else 8192 if coder == "book" else 1024)
    if coder == "fine":
        p.set_huffman_fine(b)
    p.connect(b, a, "codes")
    p.set_dims(n, 1, 1)
    p.finalize()
    return p


@pytest.mark.parametrize("n", [1, 63, 767, 769, 4096, 4097, 16_385, 300_001])
@pytest.mark.parametrize("cb", [1, 2, 4])
@pytest.mark.parametrize("coder", ["rle", "coarse", "fine", "book"])
def test_stream_in_both_buffers(fzh, coder, cb, n):
    rng = np.random.default_rng(n + cb)
    x = np.round(np.cumsum(rng.integers(-1, 2, n) * (rng.random(n) < 0.4)) * 0.02 % 1.6, 2).astype(np.float32)
    x[:: max(1, n // 7)] += 1
    d_x = fzh.DeviceBuffer.from_array(x)
    with _pipe(n, coder, cb) as p:
        ptr, size = p.compress(d_x, x.nbytes)
        want = np.empty(size, np.uint8)
        fzh.call("fzh_memcpy_dtoh", want.ctypes.data, ptr, size)
        cap = (p.max_compressed_size(x.nbytes) + x.nbytes + 15) // 16 * 16
        guard = np.full(cap + 64, 0xA5, np.uint8)
        for at in (None, 0, (size // 2 + 15) // 16 * 16):
            start = guard.copy()
            if at is not None:
                start[at:at + x.nbytes] = x.view(np.uint8)
            d_out = fzh.DeviceBuffer.from_array(start)
            src = d_x if at is None else d_out.ptr + at
            assert p.compress_into(src, x.nbytes, d_out, cap) == size
            got = d_out.download(np.uint8, guard.size)
            assert np.array_equal(got[:size], want)
            assert (got[cap:] == 0xA5).all()
            # the pool's own copy is whole too
            fzh.call("fzh_memcpy_dtoh", got.ctypes.data, ptr, size)
            assert np.array_equal(got[:size], want)
