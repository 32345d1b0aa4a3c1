"""Outlier and patch lists that an encoder's launch places: RZE containers
against the same chain with its stages unfused and bit packing of a detected
width against a given one (which place the lists in a launch of their own), the
RLE chain's lists against those, for each code width, both value types, tile
counts around a workgroup's 128 and past the limit of the kernel's own sums,
graph replays, and a chain whose indices feed another stage."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pipe(dims, coder, cb=2, dtype="f32", strict=False, fused=True, index_stage=False):
    from fzgpumodules_amd.pipeline import Pipeline
    p = Pipeline(int(np.prod(dims)) * (8 if dtype == "f64" else 4))
    if dtype == "quantizer":
        a = p.add_quantizer(1e-3, mode="ABS", quant_radius=100 if cb == 1 else 512, outlier_capacity=0.5, zigzag=True,
                            code_bytes=cb)
    else:
        a = p.add_lorenzo(1e-3, mode="ABS", quant_radius=100 if cb == 1 else 512, outlier_capacity=0.5, zigzag=True,
                          code_bytes=cb, dtype=dtype)
    if strict:
        p.set_strict(a, True, 0.2)
    if coder == "bitshuffle":
        b = p.add_bitshuffle(16384, cb)
        p.connect(b, a, "codes")
        p.connect(p.add_rze(16384, 4), b)
    elif coder == "rze":
        p.connect(p.add_rze(16384, 4), a, "codes")
    elif coder == "rle":
        p.connect(p.add_rle(cb), a, "codes")
    else:
        p.connect(p.add_bitpack(cb, 0 if coder == "pack" else 8 * cb), a, "codes")
    if index_stage:
        p.connect(p.add_rle(4), a, "outlier_indices")
    p.set_dims(*dims)
    p.set_stage_fusion(fused)
    p.finalize()
    return p


def _field(dims, dtype):
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n, np.float32) * np.float32(1e-3)).astype(np.float64 if dtype == "f64" else np.float32)
    x[rng.integers(0, n, n // 50 + 1)] = 40.0
    x[-1] = 0.0  # no outlier in the padding after it, which only the RZE chains have
    return x


def _slots(blob):
    n = int(blob[:4].view(np.uint32)[0])
    sizes = np.frombuffer(blob[4:4 + 8 * n].tobytes(), np.uint64).astype(int)
    at, out = (4 + 8 * n + 15) // 16 * 16, []
    for s in sizes:
        out.append(blob[at:at + s].tobytes())
        at += (s + 15) // 16 * 16
    return out


SHAPES = [(5, 1, 1), (1024 * 127 + 9, 1, 1), (1024 * 128, 1, 1), (1024 * 129, 1, 1), (403, 97, 1), (61, 45, 33)]
STRICT = ("bitshuffle", 2, "f32", True)
KINDS = [("rze", 2, "f32", False), ("bitshuffle", 1, "f32", False), STRICT, ("bitshuffle", 2, "f64", False),
         ("bitshuffle", 4, "f64", False)]


@pytest.mark.parametrize("dims,kind", [(d, k) for d in SHAPES for k in KINDS] +
                         [((256, 256, 256), STRICT), ((256, 264, 256), STRICT)])
def test_lists_with_the_encoder(dims, kind):
    coder, cb, dtype, strict = kind
    x = _field(dims, dtype)
    blobs = []
    for fused in (True, False):
        with _pipe(dims, coder, cb, dtype, strict, fused) as p:
            blobs.append(p.compress_array(x))
    assert np.array_equal(blobs[0], blobs[1])
    with _pipe(dims, "rle", cb, dtype, strict) as p:
        assert _slots(p.compress_array(x))[1:] == _slots(blobs[0])[1:]


@pytest.mark.parametrize("dims", SHAPES)
@pytest.mark.parametrize("cb,dtype,strict", [(1, "quantizer", False), (2, "quantizer", False), (4, "quantizer", False),
                                             (1, "f32", False), (2, "f32", True), (4, "f64", False)])
def test_lists_with_the_code_maximum(dims, cb, dtype, strict):
    x = _field(dims, dtype)
    x[:] = np.where(np.abs(x) > 1, x, 0.06 * x)  # codes below 2^8
    lists = []
    for coder in ("pack", "fixed"):
        with _pipe(dims, coder, cb, dtype, strict) as p:
            blob = p.compress_array(x)
            lists.append(_slots(blob)[1:])
            y = p.decompress_array(blob, x.dtype)[:x.size]
            assert np.abs(y.astype(np.float64) - x).max() <= 1.01e-3
    assert lists[0] == lists[1]


@pytest.mark.parametrize("strict", [False, True])
def test_graph_replays(strict):
    from fzgpumodules_amd import _fzh
    dims = (403, 97, 1)
    x = _field(dims, "f32")
    with _pipe(dims, "bitshuffle", strict=strict, fused=False) as p:
        want = p.compress_array(x)
    d = _fzh.DeviceBuffer.from_array(x)
    with _pipe(dims, "bitshuffle", strict=strict) as p:
        p.enable_graph_mode(True)
        for _ in range(5):
            ptr, n = p.compress(d, x.nbytes)
            got = np.empty(n, np.uint8)
            _fzh.call("fzh_memcpy_dtoh", got.ctypes.data, ptr, n)
            assert np.array_equal(got, want)


def test_indices_that_feed_a_stage():
    dims = (403, 97, 1)
    x = _field(dims, "f32")
    with _pipe(dims, "bitshuffle", index_stage=True) as p:
        blob = p.compress_array(x)
        y = p.decompress_array(blob, np.float32)[:x.size]
    assert np.abs(y.astype(np.float64) - x).max() <= 1.01e-3
