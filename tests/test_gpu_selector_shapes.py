"""The selector's front kernels at the edges of their loops: features of chunks
narrower, wider and smaller than a workgroup's step, chunk copies of 16-byte
and of ragged rows, and forwards of batches around a workgroup's samples."""
import numpy as np
import pytest

from fzgpumodules_amd import selector as S
from fzgpumodules_amd._fzh import DeviceBuffer, call
from oracle import selector_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1), (1, 300), (300, 1), (3, 7), (5, 255), (4, 257), (3, 1000), (256, 256),
                                   (9, 7, 5), (40, 1, 1), (500, 3, 2), (2, 2, 513), (32, 32, 32)])
def test_features_of_odd_chunks(shape):
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((3, *shape)).astype(np.float32)
    x[0] = np.round(x[0])
    x[1] *= 1e4
    eb = np.array([1e-2, 1e-3, 1e-4], np.float32)
    d_x, d_eb = DeviceBuffer.from_array(x), DeviceBuffer.from_array(eb)
    got = S.features(d_x.ptr, 3, shape, d_eb.ptr).download(np.float32, 96).reshape(3, 32)
    for i in range(3):
        # the sums' order differs from the reference's: float rounding of the features
        np.testing.assert_allclose(got[i], R.features(x[i], eb[i]), rtol=2e-6, atol=2e-6)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("field,chunk", [((48, 64), (12, 16)), ((20, 30), (4, 6)), ((8, 15, 21), (4, 5, 7)),
                                         ((4, 6, 20), (2, 3, 4)), ((9, 1), (3, 1)), ((8, 8, 8), (8, 8, 8))])
def test_chunk_copies(field, chunk, off):
    f3, c3 = (1,) * (3 - len(field)) + field, (1,) * (3 - len(chunk)) + chunk
    n = int(np.prod(field))
    x = np.arange(n + off, dtype=np.float32)
    d_x, d_c, d_y = DeviceBuffer.from_array(x), DeviceBuffer(4 * n), DeviceBuffer.from_array(np.zeros(n + off, np.float32))
    call("fzs_gather_chunks", None, d_x.ptr + 4 * off, *f3[::-1], *c3[::-1], d_c.ptr)
    g = [a // b for a, b in zip(f3, c3)]
    want = x[off:].reshape(g[0], c3[0], g[1], c3[1], g[2], c3[2]).transpose(0, 2, 4, 1, 3, 5)
    assert np.array_equal(d_c.download(np.float32, n), want.ravel())
    call("fzs_scatter_chunks", None, d_c.ptr, *f3[::-1], *c3[::-1], d_y.ptr + 4 * off)
    assert np.array_equal(d_y.download(np.float32, n + off)[off:], x[off:])


@pytest.mark.parametrize("n", [1, 3, 4, 5, 257])
def test_forward_batch_sizes(n):
    rng = np.random.default_rng(n)
    p = (rng.standard_normal(R.NP) * 0.25).astype(np.float32)
    norm = np.concatenate([rng.standard_normal(32) * 0.2, 0.5 + rng.random(32)]).astype(np.float32)
    feat = (rng.standard_normal((n, 32)) * 3).astype(np.float32)
    sel = S.Selector()
    try:
        sel.set_params(p)
        sel.norm.upload(norm)
        d_f = DeviceBuffer.from_array(feat)
        np.testing.assert_array_equal(sel.forward(d_f.ptr, n), R.forward(p, norm, feat, "exact32")[0])
    finally:
        sel.close()


@pytest.mark.parametrize("n", [4095, 4096, 4097, 8449])  # by waves up to 4096, then by threads
def test_forward_around_the_choice(n):
    test_forward_batch_sizes(n)


def test_forward_time_of_many_samples():
    """65536 samples take about as long as 4096 (60 and 51 us; 730 by waves)."""
    from fzgpumodules_amd._fzh import Event, synchronize
    sel = S.Selector()
    d_f, d_z = DeviceBuffer.zeros(65536 * 128), DeviceBuffer(65536 * 16)
    try:
        best = {}
        for n in (4096, 65536):
            best[n] = 1e9
            for _ in range(8):
                a, b = Event(), Event()
                a.record()
                call("fzs_mlp_forward", None, sel.params.ptr, sel.norm.ptr, d_f.ptr, n, d_z.ptr)
                b.record()
                synchronize()
                best[n] = min(best[n], a.elapsed_ms(b))
    finally:
        sel.close()
    assert best[65536] < 4 * best[4096]
