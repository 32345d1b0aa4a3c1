"""Performance cases: the compressor as a program on one MI355X uses it.

Every case is one call of a public entry point on data that is already on the
GPU: ``Pipeline.compress_into`` / ``Pipeline.decompress_into`` of a stage chain,
``Batch.compress`` of many fields and the gather of their results,
``SelectingCompressor.compress`` of a field whose chunks choose their chain.
The program owns the result buffers (zeroed once, as large as a result can
get); a compressed result is such a buffer and the bytes used of it.  Inputs are seeded synthetic scientific
fields (sums of sinusoids, Gaussian random fields with a power-law spectrum,
spikes, exact zeros), made on the GPU.

``listed()`` holds fixed cases, ``draw(rng)`` one more of the same ranges.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from fzgpumodules_amd import selector as sel
from fzgpumodules_amd._fzh import DeviceBuffer, call
from fzgpumodules_amd.batch import Batch
from fzgpumodules_amd.pipeline import Pipeline

DEV = "cuda"
COPY = np.dtype([("src", np.uint64), ("dst", np.uint64), ("bytes", np.uint64)])  # fzh_copy_desc


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _pipe(name, op, chain, field, nx, ny=1, nz=1, dtype="f32", mode="REL", eb=1e-3, radius=32768, capacity=0.1,
          zigzag=True, strict=True):
    return {"name": name, "kind": "pipeline", "op": op, "chain": chain, "field": field, "nx": nx, "ny": ny, "nz": nz,
            "dtype": dtype, "mode": mode, "eb": eb, "radius": radius, "capacity": capacity, "zigzag": zigzag,
            "strict": strict}


def listed():
    return [
        # one level of a climate model's cloud fraction, 1800 x 3600: the
        # command line's default chain at its default bound, both directions
        _pipe("cloud2d-compress", "compress", "bitshuffle-rze", "cloud", 3600, 1800),
        _pipe("cloud2d-decompress", "decompress", "bitshuffle-rze", "cloud", 3600, 1800),
        # a long signal at an absolute bound, run-length coded
        _pipe("signal1d-compress", "compress", "rle", "sinusoid", 1 << 24, mode="ABS", eb=1e-4, capacity=0.2,
              zigzag=False),
        _pipe("signal1d-decompress", "decompress", "rle", "sinusoid", 1 << 24, mode="ABS", eb=1e-4, capacity=0.2,
              zigzag=False),
        # a turbulence volume with isolated spikes (many outliers), Huffman
        # coded with the command line's alphabet of 2 x radius
        _pipe("turbulence3d-compress", "compress", "huffman", "turbulence", 512, 512, 512, eb=1e-4, radius=512,
              capacity=0.2),
        _pipe("turbulence3d-decompress", "decompress", "huffman", "turbulence", 512, 512, 512, eb=1e-4, radius=512,
              capacity=0.2),
        # the smallest field a program sends through the chain by itself:
        # launches and the wait for the size are what it pays
        _pipe("small2d-compress", "compress", "bitshuffle-rze", "cloud", 400, 96),
        # one 256 KiB block of a volume read back on its own (random access)
        _pipe("block3d-decompress", "decompress", "huffman", "powerlaw", 64, 64, 16, radius=512, capacity=0.2,
              strict=False),
        # double precision simulation output with sides that no tile divides
        _pipe("ragged3d-f64-compress", "compress", "bitshuffle-rze", "powerlaw", 301, 203, 157, dtype="f64",
              radius=512, capacity=0.2, strict=False),
        # pointwise quantisation and fixed-width packing (no prediction),
        # sides that no vector width divides
        _pipe("quantized2d-compress", "compress", "quantizer-bitpack", "powerlaw", 3001, 2003, mode="ABS", eb=1e-3,
              capacity=0.2, strict=False),
        # a snapshot: many variables of uneven size and shape in one call
        {"name": "snapshot-compress", "kind": "batch", "fields": 60, "max_mib": 64, "shapes": 4, "eb": 1e-3, "strict": True},
        # a field of mixed regimes, every 256 KiB chunk with the chain that
        # the trained selector picks; the container ends in host memory
        {"name": "mixed2d-select-compress", "kind": "select", "nx": 2048, "ny": 16384, "eb": 1e-3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a chain, a direction, an element count spread over its
    logarithm from one small block to the largest listed field, a shape."""
    r = rng.random()
    if r < 0.06:
        return {"kind": "batch", "fields": rng.randint(8, 60), "max_mib": rng.choice([4, 16, 64]),
                "shapes": rng.randrange(1 << 20), "eb": rng.choice([1e-2, 1e-3, 1e-4]), "strict": rng.random() < 0.7}
    if r < 0.12:
        return {"kind": "select", "nx": 256 * rng.randint(1, 8), "ny": 512 * rng.randint(2, 32),
                "eb": rng.choice([1e-2, 1e-3])}
    op = rng.choice(["compress", "decompress"])
    chain = rng.choice(["bitshuffle-rze", "bitshuffle-rze", "rle", "huffman", "huffman", "quantizer-bitpack"])
    nd = 1 if chain == "rle" else rng.choice([1, 2, 3])
    n = _log(rng, 30000, 1 << (24 if chain in ("rle", "quantizer-bitpack") else 27 if nd == 3 else 25))
    nx, ny, nz = n, 1, 1
    if nd == 2:
        nx = min(8192, max(33, int(math.sqrt(n * math.exp(rng.uniform(-1.4, 1.4))))))
        ny = min(4096, max(2, n // nx))
    elif nd == 3:
        side = n ** (1.0 / 3.0)
        nx = min(512, max(9, int(side * math.exp(rng.uniform(-0.7, 0.7)))))
        ny = min(512, max(9, int(side * math.exp(rng.uniform(-0.7, 0.7)))))
        nz = min(512, max(2, n // (nx * ny)))
    field = {1: "sinusoid", 2: rng.choice(["cloud", "powerlaw"]), 3: rng.choice(["turbulence", "powerlaw"])}[nd]
    dtype = "f64" if chain in ("bitshuffle-rze", "huffman") and n <= 1 << 25 and rng.random() < 0.2 else "f32"
    strict = dtype == "f32" and chain != "quantizer-bitpack" and rng.random() < 0.6
    radius = 512 if chain == "huffman" or dtype == "f64" else 32768
    eb = 1e-3 if chain == "huffman" or field == "cloud" else rng.choice([1e-3, 1e-4])
    mode = "ABS" if chain in ("rle", "quantizer-bitpack") else "REL"
    c = _pipe("", op, chain, field, nx, ny, nz, dtype, mode, eb, radius, 0.2, chain != "rle", strict)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Fields
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _pow2(n):
    return 1 << max(0, int(n) - 1).bit_length()


def _power_law(shape, expo, g):
    """Gaussian random field of unit deviation, power ~ k^expo: a window of a
    periodic field whose sides are powers of two."""
    full = [_pow2(s) for s in shape]
    f = torch.fft.rfftn(torch.randn(full, generator=g, device=DEV, dtype=torch.float32))
    k2 = 0
    for ax, n in enumerate(full):
        k = torch.fft.rfftfreq(n, device=DEV) if ax == len(full) - 1 else torch.fft.fftfreq(n, device=DEV)
        k2 = k2 + (k * k).reshape([-1 if a == ax else 1 for a in range(len(full))])
    k2.view(-1)[0] = 1.0
    k2 = k2 ** (expo / 4.0)
    k2.view(-1)[0] = 0.0
    f = torch.fft.irfftn(f * k2, s=full)
    f = f[tuple(slice(0, s) for s in shape)]
    return f / f.std()


def _field(case, seed):
    g = _gen(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    shape = [s for s in (nz, ny, nx) if s > 1]
    dt = torch.float64 if case["dtype"] == "f64" else torch.float32
    if case["field"] == "sinusoid":
        i = torch.arange(nx, device=DEV, dtype=torch.float64)
        u = torch.rand(3, 8, generator=g, device=DEV, dtype=torch.float64).cpu()
        x = 1e-3 * torch.randn(nx, generator=g, device=DEV, dtype=torch.float64)
        for k in range(8):
            freq, amp, ph = 1e-5 + u[0, k] * 1e-2, 0.1 + 0.9 * u[1, k], 2 * math.pi * u[2, k]
            x += float(amp) * torch.sin(2 * math.pi * float(freq) * i + float(ph))
    elif case["field"] == "cloud":  # ~30% exact zeros, maximum 1
        x = _power_law(shape, -3.0, g)
        s = x.reshape(-1)[:: max(1, x.numel() // 100000)]
        q = torch.quantile(s, 0.30)
        x = ((x - q) / (x.max() - q)).clamp(0.0, 1.0)
    elif case["field"] == "turbulence":  # 1% of the values are spikes
        x = _power_law(shape, -5.0 / 3.0, g).reshape(-1)
        hit = torch.rand(x.numel(), generator=g, device=DEV) < 0.01
        x = torch.where(hit, x * 100.0, x)
    else:  # smooth simulation output
        x = _power_law(shape, -4.0, g)
        if dt == torch.float64:
            x = x.double() + 1e-6 * torch.randn(shape, generator=g, device=DEV, dtype=torch.float64)
    return x.reshape(-1).to(dt).contiguous()


def _snapshot_dims(case):
    """Shapes of a snapshot's fields: sizes 64 KiB .. max_mib MiB log-uniform,
    thirds in 1D, 2D and 3D."""
    r = np.random.default_rng(case["shapes"])
    dims = []
    for i in range(case["fields"]):
        n = int(math.exp(r.uniform(math.log(16384), math.log(case["max_mib"] * 262144))))
        if i % 3 == 0:
            d = (n, 1, 1)
        elif i % 3 == 1:
            nx = min(4096, max(32, int(math.sqrt(n * math.exp(r.uniform(-1.4, 1.4))))))
            d = (nx, min(4096, max(2, n // nx)), 1)
        else:
            s = n ** (1.0 / 3.0)
            nx = min(256, max(8, int(s * math.exp(r.uniform(-0.7, 0.7)))))
            ny = min(256, max(8, int(s * math.exp(r.uniform(-0.7, 0.7)))))
            d = (nx, ny, min(256, max(2, n // (nx * ny))))
        dims.append(d)
    return dims


def _snapshot(case, seed):
    """(fields, dims): windows of power-law fields of several exponents."""
    g = _gen(seed)
    r = np.random.default_rng(seed)
    expos = (-1.5, -3.0, -4.5)
    base = {}
    side = {1: (1 << 24,), 2: (4096, 4096), 3: (256, 256, 256)}
    out, dims = [], _snapshot_dims(case)
    for i, d in enumerate(dims):
        nd = i % 3 + 1
        key = (nd, expos[int(r.integers(3))])
        if key not in base:
            base[key] = _power_law(side[nd], key[1], g)
        win = []
        for full, want in zip(side[nd], d[:nd][::-1]):
            o = int(r.integers(full - want + 1))
            win.append(slice(o, o + want))
        out.append(base[key][tuple(win)].clone().reshape(-1))
    return out, dims


def _mixed(nx, ny, seed):
    """Bands of 256 rows: smooth, noise, 80% zeros, piecewise constant, counts."""
    g = _gen(seed)
    bands = []
    for b in range(ny // 256):
        k = b % 5
        if k == 0:
            x = _power_law((256, nx), -4.0, g)
        elif k == 1:
            x = torch.randn(256, nx, generator=g, device=DEV)
        elif k == 2:
            x = torch.randn(256, nx, generator=g, device=DEV)
            x = torch.where(torch.rand(256, nx, generator=g, device=DEV) < 0.8, torch.zeros_like(x), x)
        elif k == 3:
            x = torch.randn(8, nx // 64, generator=g, device=DEV).repeat_interleave(32, 0).repeat_interleave(64, 1)
        else:
            x = torch.poisson(torch.full((256, nx), 20.0, device=DEV), generator=g)
        bands.append(x)
    return torch.cat(bands).float().contiguous()


def _model(seed):
    """Selector weights: a short training on labelled chunks of its own."""
    n = 320
    x = _mixed(256, 256 * n, seed + 77)
    eb = torch.full((n,), float(np.float32(1e-3) * np.float32(x.abs().max().item())), device=DEV)
    torch.cuda.synchronize()
    f = sel.features(x.data_ptr(), n, (256, 256), eb.data_ptr())
    feat = f.download(np.float32, 32 * n).reshape(n, 32)
    sizes = sel.label_sizes(x.data_ptr(), n, (256, 256), eb.data_ptr())
    m = sel.Selector(seed=11)
    m.fit(feat, sel.regret_costs(sizes), epochs=20, batch=64)
    p, q = m.get_params(), m.get_norm()
    m.close()
    f.free()
    return p, q


# ---------------------------------------------------------------------------
# The calls
# ---------------------------------------------------------------------------
def _chain(c):
    n = c["nx"] * c["ny"] * c["nz"]
    p = Pipeline(n * (8 if c["dtype"] == "f64" else 4))
    if c["chain"] == "quantizer-bitpack":
        first = p.add_quantizer(c["eb"], mode=c["mode"], quant_radius=c["radius"], outlier_capacity=c["capacity"],
                                zigzag=c["zigzag"])
        last = p.add_bitpack(2, 0)
        p.connect(last, first, "codes")
    else:
        first = p.add_lorenzo(c["eb"], mode=c["mode"], quant_radius=c["radius"], outlier_capacity=c["capacity"],
                              zigzag=c["zigzag"], dtype=c["dtype"])
        if c["strict"]:
            p.set_strict(first, True)
        if c["chain"] == "rle":
            p.connect(p.add_rle(2), first, "codes")
        elif c["chain"] == "huffman":
            p.connect(p.add_huffman(2, 2 * c["radius"]), first, "codes")
        else:
            bs = p.add_bitshuffle(16384, 2)
            p.connect(bs, first, "codes")
            p.connect(p.add_rze(16384, 4), bs)
    p.set_dims(c["nx"], c["ny"], c["nz"])
    p.finalize()
    return p


def prepare(case, seed):
    if case["kind"] == "batch":
        fields, dims = _snapshot(case, seed)
        torch.cuda.synchronize()
        b = Batch(case["eb"], "REL", 32768, 0.1, True, strict=case["strict"])
        b.set_fields([(f.data_ptr(), d) for f, d in zip(fields, dims)])
        out = torch.zeros(sum(f.numel() for f in fields) * 8 + (len(fields) << 16), dtype=torch.uint8, device=DEV)
        return {"case": case, "fields": fields, "batch": b, "out": out,
                "copies": np.zeros(len(fields), COPY), "d_copies": DeviceBuffer(COPY.itemsize * len(fields))}
    if case["kind"] == "select":
        x = _mixed(case["nx"], case["ny"], seed)
        sc = sel.SelectingCompressor((256, 256))
        sc.set_model(*_model(seed))
        torch.cuda.synchronize()
        return {"case": case, "x": x, "sc": sc, "out": np.zeros(2 * x.nbytes, np.uint8)}
    x = _field(case, seed)
    torch.cuda.synchronize()
    p = _chain(case)
    st = {"case": case, "x": x, "pipe": p}
    if case["op"] == "decompress":
        blob = torch.empty(p.max_compressed_size(x.nbytes), dtype=torch.uint8, device=DEV)
        n = p.compress_into(x.data_ptr(), x.nbytes, blob.data_ptr(), blob.numel())
        st["blob"], st["y"] = blob[:n].clone(), torch.empty_like(x)
        del st["x"]
    else:
        st["out"] = torch.zeros(p.max_compressed_size(x.nbytes), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    return st


def run(state):
    case = state["case"]
    stream = torch.cuda.current_stream().cuda_stream
    if case["kind"] == "batch":
        # results back to back in the program's buffer
        b, out, cp = state["batch"], state["out"], state["copies"]
        b.compress(stream)
        base, _ = b.output()
        pos, dst = 0, out.data_ptr()
        for i in range(b.n):
            off, nb = b.field_result(i)
            cp[i] = (base + off, dst + pos, nb)
            pos += (nb + 15) & ~15
        if pos > out.numel():
            raise RuntimeError("result buffer too small")
        state["d_copies"].upload(cp)
        call("fzh_gather", stream, state["d_copies"].ptr, b.n)
        return {"data": out, "bytes": cp["bytes"].copy()}
    if case["kind"] == "select":
        blob = state["sc"].compress(state["x"].data_ptr(), (case["ny"], case["nx"]), case["eb"], sel.LEARNED,
                                    stream=stream)
        state["out"][:blob.size] = blob
        return {"data": state["out"], "bytes": blob.size}
    p = state["pipe"]
    if case["op"] == "decompress":
        blob, y = state["blob"], state["y"]
        p.decompress_into(blob.data_ptr(), blob.numel(), y.data_ptr(), y.nbytes, stream)
        return y
    x, out = state["x"], state["out"]
    n = p.compress_into(x.data_ptr(), x.nbytes, out.data_ptr(), out.numel(), stream)
    return {"data": out, "bytes": n}


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how results are compared
# ---------------------------------------------------------------------------
# input bytes over compressed bytes that the fields reach, typically
RATIO = {"bitshuffle-rze": 8.0, "rle": 0.7, "huffman": 3.6, "quantizer-bitpack": 2.0, "batch": 6.0, "select": 8.0}


def work(case):
    if case["kind"] == "batch":
        raw, ratio = 4 * sum(x * y * z for x, y, z in _snapshot_dims(case)), RATIO["batch"]
    elif case["kind"] == "select":
        raw, ratio = 4 * case["nx"] * case["ny"], RATIO["select"]
    else:
        raw = case["nx"] * case["ny"] * case["nz"] * (8 if case["dtype"] == "f64" else 4)
        ratio = RATIO[case["chain"]] * (2.0 if case["dtype"] == "f64" else 1.0)
    # a prediction from neighbours, a rounding and a code per value
    return {"bytes": int(raw + raw / ratio), "flops": int(8 * raw / 4)}


def tolerance(case):
    # the streams are a format, and a strict bound's patches belong to the
    # exact values that the decoder reconstructs
    return "exact"


def exact(case, seed):
    """The values a decoder gives back: whole multiples of twice the bound,
    original values where that misses the bound under the strict setting."""
    if case["kind"] != "pipeline" or case["op"] != "decompress":
        return None
    x = _field(case, seed)
    dt = np.float64 if case["dtype"] == "f64" else np.float32
    eb = dt(np.float32(case["eb"]))
    if case["mode"] == "REL":
        eb = dt(eb * dt(np.float32(x.abs().max().item())))
    r = dt(dt(1) / (dt(2) * eb))
    v = (x * float(r)).double()  # the product is the format's, at the input's precision
    if case["chain"] == "quantizer-bitpack":
        q = torch.round(v)
    else:  # halves go away from zero
        q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    y = q * (2.0 * float(eb))
    if case["chain"] == "quantizer-bitpack":
        y = torch.where(q.abs() < case["radius"], y, x.double())
    if case["strict"]:
        y = torch.where((q.to(x.dtype) * float(dt(2) * eb) - x).abs() > float(eb), x.double(), y)
    return y
