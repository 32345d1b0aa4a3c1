"""Which outlier lists the inverse takes as ordered: entries past the tiles'
region at the list's end (the padding's outlier of a 1D field decompressed to its
own length) leave a list in order, anywhere else they send it through the
counting sort, and either way they are dropped.  The result is that of the same
call without them (exact); the flag is the last 256-byte block of the inverse
workspace."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inverse(codes, n, dims, err, idx, ebx2):
    """(result, list taken as unordered)"""
    from fzgpumodules_amd._fzh import DeviceBuffer, call, lib, workspace
    f64 = err.dtype == np.float64
    name = "f64" if f64 else "f32"
    dc, de, di = DeviceBuffer.from_array(codes), DeviceBuffer.from_array(err), DeviceBuffer.from_array(idx)
    dn = DeviceBuffer.from_array(np.array([idx.size], np.uint32))
    out = DeviceBuffer.zeros(n * err.itemsize)
    size = lib().fzh_lorenzo_quant_inv_f64_ws_bytes if f64 else lib().fzh_lorenzo_quant_inv_ws_bytes
    ws = workspace(size(n, *dims, idx.size))
    call(f"fzh_lorenzo_quant_inv_{name}", None, dc.ptr, n, *dims, de.ptr, di.ptr, dn.ptr, idx.size,
         float(ebx2), 1, 2, out.ptr, ws.ptr, ws.nbytes)
    return out.download(err.dtype, n), bool(ws.download(np.uint32, 1, ws.nbytes - 256)[0])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [5_000, 9_215, 9_217, 1_000_001])
def test_padded_1d_field(gpu, dtype, n):
    padded = -(-n // 8192) * 8192
    x = np.zeros(padded, dtype)
    rng = np.random.default_rng(n)
    x[:n] = np.cumsum(rng.integers(-3, 4, n))
    x[rng.choice(n, 400, replace=False)] += 2000
    x[n - 1] = 3000  # and zeros behind it
    fwd = gpu.lorenzo_fwd if dtype == np.float32 else gpu.lorenzo_fwd64
    codes, err, idx, cnt = fwd(x, (padded, 1, 1), 1.0, 512, True, 2)
    assert cnt == idx.size > 256 and idx[-1] >= n
    y, unordered = _inverse(codes, n, (n, 1, 1), err, idx, 1.0)
    assert np.array_equal(y, x[:n])
    assert not unordered


@pytest.mark.parametrize("dims", [(5_000, 1, 1), (203, 101, 1), (33, 17, 29)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("where", ["end", "middle", "start", "all", "swapped"])
def test_entries_outside(gpu, dims, dtype, where):
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    x = np.cumsum(rng.integers(-3, 4, n)).astype(dtype)
    x[rng.choice(n, 700, replace=False)] += 2000
    fwd = gpu.lorenzo_fwd if dtype == np.float32 else gpu.lorenzo_fwd64
    codes, err, idx, cnt = fwd(x, dims, 1.0, 512, True, 2)
    assert cnt > 300
    out = np.array([n, n + 5, 0xFFFFFFFF, n + 1], np.uint32)
    if where == "all":
        codes = np.zeros_like(codes)
        want = np.zeros(n, dtype)
        err, idx = np.full(300, 7, dtype), np.tile(out, 75)
    else:
        want = x
        if where == "swapped":
            o = np.r_[np.arange(200, idx.size), np.arange(200)]
            err, idx = err[o], idx[o]
        else:
            at = {"end": idx.size, "middle": idx.size // 2, "start": 0}[where]
            err, idx = np.insert(err, at, np.full(4, 9, dtype)), np.insert(idx, at, out)
    y, unordered = _inverse(codes, n, dims, err, idx, 1.0)
    assert np.array_equal(y, want)
    assert unordered == (where in ("middle", "start", "swapped"))
