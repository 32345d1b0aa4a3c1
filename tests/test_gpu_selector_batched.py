"""The selector's batched chains: every chunk's bytes in the container equal
fz::Pipeline::compress of that chunk alone, the container's checksum equals
zlib's over the same bytes, and the container decodes -- over chunk shapes of
1, 2 and 3 dimensions (a single partition of the Huffman stream to hundreds),
constant chunks (a codebook of one symbol), dense outliers past a tile's list
slots, one chunk (not batched), and new fields on one handle."""
import zlib

import numpy as np
import pytest

from fzgpumodules_amd import fields
from fzgpumodules_amd import selector as S
from fzgpumodules_amd._fzh import DeviceBuffer

pytestmark = pytest.mark.gpu

SHAPES = [((4096,), 9), ((64, 64), 13), ((256, 256), 6), ((16, 64, 64), 3), ((8, 24, 64), 5), ((3, 20, 4096), 2),
          ((64, 64), 1), ((64, 64), 2)]


def _field(shape, n, kind, seed):
    """n chunks of `shape` stacked along the slowest axis."""
    rng = np.random.default_rng(seed)
    c = np.zeros((n,) + shape, np.float32)
    for i in range(n):
        k = i % 4 if kind == "mixed" else kind
        if k == 0:  # smooth
            c[i] = np.cumsum(0.002 * rng.standard_normal(shape), axis=-1)
        elif k == 1:  # a few large values (outliers), one tile full of them
            c[i] = 0.001 * rng.standard_normal(shape)
            flat = c[i].reshape(-1)
            flat[rng.integers(0, flat.size, flat.size // 300)] = 3
            flat[:40:2] = 4
        elif k == 2:  # constant
            c[i] = 0.25
        else:  # noise over much of the alphabet
            c[i] = 0.3 * rng.standard_normal(shape)
    return c.reshape((n * shape[0],) + shape[1:])


def _parse(blob, n):
    """(per-chunk blobs, choices) of an FZS1 container."""
    mask = int(blob[64:68].view(np.uint32)[0])
    o = 68
    rec = None
    # the stage records end where the choices, the sizes and the padded
    # results exactly fill the rest
    for end in range(o, min(blob.size, 68 + 4 * 4 + 12 * 512), 4):
        oc, ob = end, end + (n + 7) // 8 * 8
        if ob + 8 * n > blob.size:
            break
        sizes = blob[ob:ob + 8 * n].copy().view(np.uint64).astype(np.int64)
        if (blob[oc:oc + n] < 4).all() and (sizes > 0).all() and ob + 8 * n + ((sizes + 15) // 16 * 16).sum() == blob.size:
            rec = (oc, ob + 8 * n, sizes)
    assert mask and rec
    oc, p, sizes = rec
    out = []
    for s in sizes:
        out.append(blob[p:p + s])
        p += (s + 15) // 16 * 16
    return out, blob[oc:oc + n]


# the Huffman chain is batched from 4 chunks on, with codebooks of the host up to 64
HUFFMAN = [((4096,), 4), ((64, 64), 3), ((64, 64), 5), ((4096,), 64), ((64, 64), 65), ((8, 24, 64), 67),
           ((256, 256), 41), ((16, 64, 64), 4), ((3, 20, 4096), 18)]


@pytest.mark.parametrize("chain,shape,n", [(c, *x) for c in (1, 2) for x in SHAPES] + [(2, *x) for x in HUFFMAN])
def test_chunks_equal_the_pipeline(shape, n, chain):
    sc = S.SelectingCompressor(shape)
    try:
        for kind, seed in (("mixed", 1), (2, 2), ("mixed", 3), ("mixed", 3), (1, 4)):  # new plans, a kept one
            x = _field(shape, n, kind, seed)
            d = DeviceBuffer.from_array(x)
            blob = sc.compress(d.ptr, x.shape, 1e-3, mode=S.FIXED, chain=chain)
            got, choice = _parse(blob, n)
            assert (choice == chain).all()
            assert int(blob[60:64].view(np.uint32)[0]) == zlib.crc32(blob[64:].tobytes())
            eb = float(blob[56:60].view(np.float32)[0])
            with S.chain_pipeline(chain, eb, shape) as p:
                for i, ch in enumerate(x.reshape((n,) + shape)):
                    want = p.compress_array(np.ascontiguousarray(ch))
                    assert np.array_equal(got[i], want), (kind, i)
            y = DeviceBuffer(x.nbytes)
            sc.decompress(blob, y.ptr, x.size)
            err = np.abs(y.download(np.float32, x.size).astype(np.float64) - x.reshape(-1)).max()
            assert err <= eb * 1.001
            d.free()
            y.free()
    finally:
        sc.close()


def test_all_chains_in_one_container():
    """Chunks of five regimes under the exhaustive choice: batched and single
    chunks interleave in one container."""
    shape, n = (256, 256), 25
    x = np.concatenate([fields.regime_field(i % 5, shape, 40 + i) for i in range(n)])
    d = DeviceBuffer.from_array(x)
    sc = S.SelectingCompressor(shape)
    blob = sc.compress(d.ptr, x.shape, 1e-3, mode=S.EXHAUSTIVE)
    got, choice = _parse(blob, n)
    assert np.array_equal(choice, sc.choices()) and len(set(choice.tolist())) >= 2
    assert int(blob[60:64].view(np.uint32)[0]) == zlib.crc32(blob[64:].tobytes())
    eb = float(blob[56:60].view(np.float32)[0])
    for i, ch in enumerate(x.reshape((n,) + shape)):
        with S.chain_pipeline(int(choice[i]), eb, shape) as p:
            assert np.array_equal(got[i], p.compress_array(np.ascontiguousarray(ch))), (i, choice[i])
    sc.close()
    d.free()


@pytest.mark.parametrize("n,most", [(2, 3), (8, 3), (32, 2)])
def test_time_of_a_few_huffman_chunks(n, most):
    """Noisy chunks in 0.5, 0.8 and 1.1 ms (the quantizer's chain 0.4, 0.8 and 1.7); 3.1 to 3.4 with
    codebooks built by one lane each."""
    import time
    from fzgpumodules_amd._fzh import synchronize
    x = np.random.default_rng(2).standard_normal((256 * n, 256)).astype(np.float32)
    d = DeviceBuffer.from_array(x)
    sc = S.SelectingCompressor((256, 256))
    best = {}
    for chain in (2, 3):
        best[chain] = 1e9
        for _ in range(12):
            synchronize()
            t = time.perf_counter()
            sc.compress(d.ptr, x.shape, 1e-3, mode=S.FIXED, chain=chain)
            best[chain] = min(best[chain], time.perf_counter() - t)
    sc.close()
    d.free()
    print(n, best)
    assert best[2] < most * best[3]


def test_batch_without_memory():
    """A field whose batch does not fit the memory that is left: the same container
    through pipelines, whose scratch is that of a chunk."""
    import ctypes as C
    from fzgpumodules_amd._fzh import lib
    x = np.cumsum(np.random.default_rng(1).standard_normal((256 * 256, 256)) * 0.01, axis=1).astype(np.float32)
    d = DeviceBuffer.from_array(x)  # 64 MiB; the batch takes 170
    blobs = []
    for leave in (None, 110 << 20):
        sc = S.SelectingCompressor((256, 256))
        if leave is not None:
            sc.compress(d.ptr, (256 * 3, 256), 1e-3, mode=S.FIXED, chain=2)  # the handle's streams and pipelines
            full = []
            for _ in range(4):  # (the free size that is reported is coarse next to a large buffer)
                free, total = C.c_size_t(), C.c_size_t()
                assert lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
                if free.value > leave + x.nbytes + (8 << 20):
                    full.append(DeviceBuffer(free.value - leave - x.nbytes))
        blobs.append(sc.compress(d.ptr, x.shape, 1e-3, mode=S.FIXED, chain=2))
        sc.close()
    for b in [*full, d]:
        b.free()
    assert np.array_equal(*blobs)
