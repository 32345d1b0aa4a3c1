"""A caller's buffer that shares memory with a call's input: decompress with
the compressed bytes at the start, in the middle and at the end of the output
buffer, byte for byte the result of separate buffers.  Sizes that a chain pads
and that it doesn't, outlier and patch lists short enough for the inverse
kernel to read itself (256) and longer ones, a chain with one output, buffers
of exactly the original size and with room for the padding.  Compress with the
input inside the output buffer, where a call that fails leaves the input."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fzh():
    from fzgpumodules_amd import _fzh
    return _fzh


def _pipe(chain, dims, dtype, strict):
    from fzgpumodules_amd.pipeline import Pipeline
    n = int(np.prod(dims))
    p = Pipeline(n * (8 if dtype == "f64" else 4))
    if chain == "plain":  # one output
        b = p.add_bitshuffle(16384, 2)
        p.connect(p.add_rze(16384, 4), b)
    elif chain == "pack":
        a = p.add_quantizer(1e-3, mode="ABS", zigzag=True, outlier_capacity=0.3)
        p.connect(p.add_bitpack(2, 0), a, "codes")
    else:
        a = p.add_lorenzo(1e-3, mode="ABS", quant_radius=512, outlier_capacity=0.3, zigzag=True, dtype=dtype)
        if strict:
            p.set_strict(a, True, 1.0)
        if chain == "rze":
            b = p.add_bitshuffle(16384, 2)
            p.connect(b, a, "codes")
            p.connect(p.add_rze(16384, 4), b)
        elif chain == "huffman":
            p.connect(p.add_huffman(2, 1024), a, "codes")
        else:
            p.connect(p.add_rle(2), a, "codes")
    p.set_dims(*dims)
    p.finalize()
    return p


def _field(dims, dtype, lists):
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    x = np.cumsum(rng.standard_normal(n) * 1e-3)
    at = np.sort(rng.choice(n, 100 if lists == "short" else n // 20, replace=False))
    if lists == "short":
        x[at] += 3
    else:  # large values: the reconstruction rounds past the bound, so patches too
        x[: n // 2] += 30_000
        x[at] += 5
    return x.astype(np.float64 if dtype == "f64" else np.float32)


CASES = [("rze", (403, 97, 1), "f32", True), ("rze", (512, 96, 1), "f32", True), ("rze", (50_001, 1, 1), "f32", True),
         ("rze", (50_001, 1, 1), "f64", False), ("rze", (33, 45, 27), "f32", True), ("huffman", (61, 45, 33), "f32", True),
         ("rle", (70_001, 1, 1), "f32", False), ("pack", (501, 203, 1), "f32", False), ("plain", (403, 97, 1), "f32", False)]


@pytest.mark.parametrize("lists", ["short", "long"])
@pytest.mark.parametrize("chain,dims,dtype,strict", CASES)
def test_decompress_over_its_input(fzh, chain, dims, dtype, strict, lists):
    x = _field(dims, dtype, lists)
    with _pipe(chain, dims, dtype, strict) as p:
        blob = p.compress_array(x)
        sizes = dict(p.outputs())
        if strict:
            assert (sizes["patch_values"] > 4 * 256) == (lists == "long")
        want = p.decompress_array(blob, x.dtype)[:x.size].view(np.uint8)
        d_b = fzh.DeviceBuffer.from_array(blob)
        for spare in (0, 1 << 15):
            cap = x.nbytes + spare
            base = (blob.size + 15) // 16 * 16  # the output lies here, so that every place below is inside the arena
            for at in (base, base + cap // 2 // 16 * 16, (base + cap - blob.size) // 16 * 16, base - base // 2 // 16 * 16):
                arena = np.full(base + cap + blob.size + 64, 0xA5, np.uint8)
                arena[at:at + blob.size] = blob
                d = fzh.DeviceBuffer.from_array(arena)
                assert p.decompress_into(d.ptr + at, blob.size, d.ptr + base, cap) == x.nbytes
                got = d.download(np.uint8, arena.size)
                assert np.array_equal(got[base:base + x.nbytes], want)
                assert (got[max(base + cap, at + blob.size):] == 0xA5).all()
                d.free()
        assert d_b.ptr


@pytest.mark.parametrize("chain", ["rze", "huffman", "rle"])
@pytest.mark.parametrize("at", [0, 4096, -1])
def test_failed_compress_leaves_its_input(fzh, chain, at):
    from fzgpumodules_amd.pipeline import Pipeline
    dims = (403, 97, 1)
    x = _field(dims, "f32", "long")
    with Pipeline(x.nbytes) as p:
        a = p.add_lorenzo(1e-3, mode="ABS", quant_radius=512, outlier_capacity=0.3, zigzag=True)
        p.set_strict(a, True, 1e-4)  # room for 4 patches
        if chain == "rze":
            b = p.add_bitshuffle(16384, 2)
            p.connect(b, a, "codes")
            p.connect(p.add_rze(16384, 4), b)
        else:
            p.connect(p.add_huffman(2, 1024) if chain == "huffman" else p.add_rle(2), a, "codes")
        p.set_dims(*dims)
        p.finalize()
        cap = (p.max_compressed_size(x.nbytes) + x.nbytes + 15) // 16 * 16
        if at < 0:
            at = (cap - x.nbytes) // 16 * 16
        start = np.full(cap + 64, 0xA5, np.uint8)
        start[at:at + x.nbytes] = x.view(np.uint8)
        d = fzh.DeviceBuffer.from_array(start)
        for _ in range(2):  # the second call runs on the first one's buffers
            with pytest.raises(fzh.FzhError, match="patch"):
                p.compress_into(d.ptr + at, x.nbytes, d, cap)
            got = d.download(np.uint8, start.size)
            assert np.array_equal(got[at:at + x.nbytes], x.view(np.uint8))
            assert (got[cap:] == 0xA5).all()
