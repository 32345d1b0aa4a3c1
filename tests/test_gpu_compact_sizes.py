"""Outlier and patch compaction at tile counts on both sides of the place
kernel's own sum of the counts (65536 counts of all lists): the lists of a
field equal the oracle's, value by value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [65535, 65536, 65537, 70_001])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_lists_over_many_tiles(tiles, dtype):
    import oracle as orc
    from fzgpumodules_amd import kernels as K
    n = tiles * 1024 - 5
    x = np.zeros(n, dtype)
    rng = np.random.default_rng(tiles)
    at = np.unique(np.r_[0, n - 1, rng.integers(0, n, 3000)])  # a few outliers, most tiles without
    x[at] = 1e6 * (1 + rng.random(at.size))
    fwd = K.lorenzo_fwd if dtype == np.float32 else K.lorenzo_fwd64
    m = 20_000
    codes, err, idx, cnt = fwd(x, (n, 1, 1), 1.0, 512, True, 2, m)
    oc, oe, oi, on = orc.lorenzo_fwd(x, (n, 1, 1), 1.0, 512, True, 2, m)
    assert cnt == on and np.array_equal(codes, oc)
    assert np.array_equal(idx, oi) and np.array_equal(err, oe)


@pytest.mark.parametrize("nz", [1016, 1024])  # two lists: 2 x 32512 and 2 x 32768 counts, then past the limit
@pytest.mark.parametrize("more", [0, 8])
def test_strict_lists_over_many_tiles(nz, more):
    from fzgpumodules_amd.pipeline import Pipeline
    nx, ny = 64, 256
    n = nx * ny * (nz + more)
    rng = np.random.default_rng(nz)
    x = np.cumsum(rng.standard_normal(n).astype(np.float32) * np.float32(0.3)).astype(np.float32)
    x[rng.integers(0, n, 2000)] = 1e5
    with Pipeline(4 * n) as p:
        lz = p.add_lorenzo(1e-3, mode="ABS", quant_radius=512, outlier_capacity=0.9, zigzag=True)
        p.set_strict(lz, True, 1.0)
        p.connect(p.add_huffman(2, 1024), lz, "codes")
        p.set_dims(nx, ny, nz + more)
        p.finalize()
        y = p.decompress_array(p.compress_array(x))
    assert np.abs(y[:n].astype(np.float64) - x).max() <= np.float32(1e-3)
