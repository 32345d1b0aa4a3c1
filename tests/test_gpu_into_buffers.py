"""compress_into / decompress_into of a caller's buffer against the pool-owned
calls, byte for byte: buffers that the last launch of a call writes itself and
buffers that get a copy (too small for any result, off alignment, the pool's
own, graph mode), padded and unpadded inputs, bytes around the result, files
written after the caller has reused its buffer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fzh():
    from fzgpumodules_amd import _fzh
    return _fzh


def _pipe(chain, dims, dtype="f32", radius=512, strict=True, mode="REL"):
    from fzgpumodules_amd.pipeline import Pipeline
    n = int(np.prod(dims))
    p = Pipeline(n * (8 if dtype == "f64" else 4))
    if chain == "pack":
        a = p.add_quantizer(1e-3, mode="ABS", zigzag=True, outlier_capacity=0.2)
        p.connect(p.add_bitpack(2, 0), a, "codes")
    else:
        a = p.add_lorenzo(1e-3, mode=mode, quant_radius=radius, outlier_capacity=0.3, zigzag=True, dtype=dtype)
        if strict and dtype == "f32":
            p.set_strict(a, True)
        if chain == "rze":
            b = p.add_bitshuffle(16384, 2)
            p.connect(b, a, "codes")
            p.connect(p.add_rze(16384, 4), b)
        elif chain == "huffman":
            p.connect(p.add_huffman(2, 2 * radius), a, "codes")
        elif chain == "rle":
            p.connect(p.add_rle(2), a, "codes")
    p.set_dims(*dims)
    p.finalize()
    return p


def _field(dims, dtype, seed=1):
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    z, y, x = np.ogrid[:nz, :ny, :nx]
    f = np.sin(x * 0.05) + np.cos(y * 0.07) * np.sin(z * 0.11 + 1) + 0.01 * rng.standard_normal((nz, ny, nx))
    f.reshape(-1)[rng.integers(0, f.size, f.size // 200)] *= 30  # outliers
    f.reshape(-1)[-1] = 25.0  # the padding after it jumps
    return f.astype(np.float64 if dtype == "f64" else np.float32).ravel()


CASES = [("rze", (400, 96, 1), "f32"), ("rze", (403, 97, 1), "f32"), ("rze", (31, 17, 23), "f64"),
         ("rze", (100_003, 1, 1), "f32"), ("rze", (50_001, 1, 1), "f64"), ("rze", (64, 64, 50), "f32"),
         ("huffman", (61, 45, 33), "f32"), ("rle", (70_001, 1, 1), "f32"), ("pack", (501, 203, 1), "f32"),
         ("rze", (3, 5, 1), "f32")]


@pytest.mark.parametrize("chain,dims,dtype", CASES)
@pytest.mark.parametrize("where", ["max", "fits", "off16", "graph"])
def test_compress_into(fzh, chain, dims, dtype, where):
    x = _field(dims, dtype)
    d_x = fzh.DeviceBuffer.from_array(x)
    with _pipe(chain, dims, dtype) as p:
        ptr, n = p.compress(d_x, x.nbytes)
        want = np.empty(n, np.uint8)
        fzh.call("fzh_memcpy_dtoh", want.ctypes.data, ptr, n)
        off = 8 if where == "off16" else 0
        cap = n if where == "fits" else p.max_compressed_size(x.nbytes)
        guard = np.full(cap + 64, 0xA5, np.uint8)
        d_out = fzh.DeviceBuffer.from_array(guard)
        if where == "graph":
            p.enable_graph_mode(True)
        for _ in range(3):
            d_out.upload(guard)
            assert p.compress_into(d_x, x.nbytes, d_out.ptr + off, cap) == n
            got = d_out.download(np.uint8, guard.size)
            assert np.array_equal(got[off:off + n], want)
            assert (got[:off] == 0xA5).all() and (got[off + cap:] == 0xA5).all()
        with pytest.raises(fzh.FzhError):
            p.compress_into(d_x, x.nbytes, d_out.ptr, n - 1)
        # the pool's own buffer as the caller's
        assert p.compress_into(d_x, x.nbytes, ptr, n) == n
        fzh.call("fzh_memcpy_dtoh", got.ctypes.data, ptr, n)
        assert np.array_equal(got[:n], want)


@pytest.mark.parametrize("chain,dims,dtype", CASES)
@pytest.mark.parametrize("spare", [0, 4, 1 << 15])
def test_decompress_into(fzh, chain, dims, dtype, spare):
    x = _field(dims, dtype)
    d_x = fzh.DeviceBuffer.from_array(x)
    with _pipe(chain, dims, dtype) as p:
        blob = p.compress_array(x)
        want = p.decompress_array(blob, x.dtype)[:x.size]
        d_b = fzh.DeviceBuffer.from_array(blob)
        for off in (0, 4):
            guard = np.full(x.nbytes + spare + 64, 0xA5, np.uint8)
            d_y = fzh.DeviceBuffer.from_array(guard)
            assert p.decompress_into(d_b, blob.size, d_y.ptr + off, x.nbytes + spare) == x.nbytes
            got = d_y.download(np.uint8, guard.size)
            assert np.array_equal(got[off:off + x.nbytes], want.view(np.uint8))
            assert (got[:off] == 0xA5).all() and (got[off + x.nbytes + spare:] == 0xA5).all()
        with pytest.raises(fzh.FzhError):
            p.decompress_into(d_b, blob.size, d_y, x.nbytes - 1)
    assert d_x.ptr


@pytest.mark.parametrize("chain", ["rze", "huffman"])
def test_file_after_the_buffer_is_reused(fzh, tmp_path, chain):
    dims = (400, 96, 1)
    x = _field(dims, "f32")
    d_x = fzh.DeviceBuffer.from_array(x)
    with _pipe(chain, dims) as p:
        d_out = fzh.DeviceBuffer(p.max_compressed_size(x.nbytes))
        n = p.compress_into(d_x, x.nbytes, d_out, d_out.nbytes)
        want = p.decompress_array(d_out.download(np.uint8, n), np.float32)[:x.size]
        p.compress_into(d_x, x.nbytes, d_out, d_out.nbytes)
        fzh.call("fzh_memset", d_out.ptr, 0, d_out.nbytes)
        p.write_file(tmp_path / "a.fzm")
        from fzgpumodules_amd.pipeline import Pipeline
        assert np.array_equal(Pipeline.decompress_file(tmp_path / "a.fzm")[:x.size], want)


def test_decompress_after_one_that_failed(fzh):
    """A decompress that throws before its inverse ran leaves nothing to the next one."""
    from fzgpumodules_amd.pipeline import Pipeline
    small, large = _field((5_001, 1, 1), "f32"), _field((70_001, 1, 1), "f32")
    with Pipeline(large.nbytes) as p:
        a = p.add_lorenzo(1e-3, mode="ABS", quant_radius=512, outlier_capacity=0.3, zigzag=True)
        b = p.add_bitshuffle(16384, 2)
        p.connect(b, a, "codes")
        p.connect(p.add_rze(16384, 4), b)
        p.finalize()
        blob = p.compress_array(small)
        d_b, d_y = fzh.DeviceBuffer.from_array(blob), fzh.DeviceBuffer(small.nbytes)
        p.set_strict(a, True)  # the stage now expects patch lists that this pipeline doesn't have
        with pytest.raises(fzh.FzhError):
            p.decompress_into(d_b, blob.size, d_y, small.nbytes)
        p.set_strict(a, False)
        y = p.decompress_array(p.compress_array(large))
        assert y.size == large.size and np.abs(y - large).max() <= 1.001e-3
