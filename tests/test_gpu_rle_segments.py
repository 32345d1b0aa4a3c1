"""RLE decode where a workgroup expands its segment of 4096 runs and where the
stream goes by output tiles: run counts at a segment's edge, elements at the
limit between the two (32768 a segment), runs across windows and segments,
runs of length zero, and a stream whose lengths do not sum to the output.
Streams are written from (values, lengths); the result is numpy's repeat."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from fzgpumodules_amd import kernels
    return kernels


def _stream(vals, lens):
    v = vals.tobytes()
    return np.frombuffer(np.uint32(len(lens)).tobytes() + v + b"\0" * (-len(v) % 4)
                         + lens.astype(np.uint32).tobytes(), np.uint8)


def _lens(kind, rng):
    r = {
        "ones_4095": lambda: np.ones(4095), "ones_4096": lambda: np.ones(4096), "ones_4097": lambda: np.ones(4097),
        "one_run": lambda: np.array([5]), "short": lambda: rng.integers(1, 4, 70_001),
        "at_limit": lambda: np.full(3 * 4096, 8),
        "over_limit": lambda: np.r_[np.full(2 * 4096, 8), 9, np.full(4095, 8)],
        "one_long": lambda: np.r_[np.ones(5000), 1_000_000, np.ones(5000)],
        "windows": lambda: np.r_[1, rng.choice([1, 2, 255, 256, 257, 511, 512, 513], 300)],
        "edge_in_segment": lambda: np.r_[np.ones(4000), np.full(96, 290)],
        "zeros": lambda: np.r_[0, 0, rng.integers(0, 3, 20_000), 0],
        "mostly_zeros": lambda: np.r_[np.zeros(4096), 7, np.zeros(4095), np.zeros(4096), 3],
    }[kind]()
    return r.astype(np.int64)


KINDS = ["ones_4095", "ones_4096", "ones_4097", "one_run", "short", "at_limit", "over_limit", "one_long", "windows",
         "edge_in_segment", "zeros", "mostly_zeros"]


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32])
@pytest.mark.parametrize("kind", KINDS)
def test_expand(gpu, dtype, kind):
    rng = np.random.default_rng(len(kind))
    lens = _lens(kind, rng)
    vals = rng.integers(0, 251, lens.size).astype(dtype)
    want = np.repeat(vals, lens)
    if lens.size > want.size:  # more runs than elements: refused
        with pytest.raises(ValueError):
            gpu.rle_dec(_stream(vals, lens), dtype, want.size)
        return
    assert np.array_equal(gpu.rle_dec(_stream(vals, lens), dtype, want.size), want)


@pytest.mark.parametrize("kind", ["short", "one_long"])
@pytest.mark.parametrize("by", [-1, 1, 5000])
def test_wrong_total(gpu, kind, by):
    rng = np.random.default_rng(1)
    lens = _lens(kind, rng)
    vals = np.arange(lens.size).astype(np.uint16)
    with pytest.raises(ValueError):
        gpu.rle_dec(_stream(vals, lens), np.uint16, int(lens.sum()) + by)


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32])
@pytest.mark.parametrize("offset", [0, 1, -1])
@pytest.mark.parametrize("kind", ["even", "one_run"])
def test_largest_starts(gpu, dtype, offset, kind):
    """A segment at the limit that begins anywhere in its first window: the largest 16-bit starts."""
    win = 64 * 16 // np.dtype(dtype).itemsize
    first = np.ones(4096, np.int64)
    first[7] += offset % win
    last = np.full(4096, 8) if kind == "even" else np.r_[np.ones(4000), 32768 - 4095, np.ones(95)]
    lens = np.r_[first, last].astype(np.int64)
    assert first.sum() <= 32768 and last.sum() == 32768
    vals = np.random.default_rng(offset + 5).integers(0, 251, lens.size).astype(dtype)
    want = np.repeat(vals, lens)
    assert np.array_equal(gpu.rle_dec(_stream(vals, lens), dtype, want.size), want)
