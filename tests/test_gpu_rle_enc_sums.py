"""RLE encode at tile counts around the write kernel's own sum of the counts
(16384 tiles, four per workgroup): the stream against numpy's runs."""
import numpy as np
import pytest

from fzgpumodules_amd._fzh import DeviceBuffer, call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5, 1023, 16384, 16385, 16389])
@pytest.mark.parametrize("more", [-1, 0, 1])
def test_streams(tiles, more):
    n = 2048 * tiles + more  # 4-byte values: 2048 a tile
    rng = np.random.default_rng(tiles)
    x = np.cumsum(rng.random(n) < 0.2).astype(np.uint32)
    x[n // 3:n // 2] = 7  # tiles without a start
    cap, ws = 8 + 8 * n + 64, 1 << 20
    d_x, d_o, d_s, d_w = DeviceBuffer.from_array(x), DeviceBuffer(cap), DeviceBuffer(16), DeviceBuffer(ws)
    for _ in range(2):
        call("fzh_rle_enc", None, d_x.ptr, n, 4, d_o.ptr, cap, d_s.ptr, d_w.ptr, ws)
        size = int(d_s.download(np.uint64, 1)[0])
        at = np.flatnonzero(np.r_[True, x[1:] != x[:-1]])
        want = np.r_[np.uint32(at.size), x[at], np.diff(np.r_[at, n]).astype(np.uint32)].astype(np.uint32)
        assert size == want.nbytes and np.array_equal(d_o.download(np.uint32, want.size), want)
