// quant_bitpack.hip — direct-value quantizer (ABS/NOA) and power-of-two bit
// packing (gfx950).
//
// Quantizer ABS/NOA (modules/quantizers/quantizer/quantizer.cu:30-67, 116-137):
//   q = __float2int_rn(x * ebx2_r)  (round half to even, saturating)
//   |q| < radius and |x| < threshold -> code = q (two's complement in TCode)
//   or zigzag(q); otherwise code 0 and an outlier (x, i).
//   inverse: out = (float)q * ebx2, then outliers assign their value.
// Outliers come out in index order: each 1024-element tile writes its list
// to a scratch slot and a compaction kernel places the lists (the reference
// appends with atomics).
// In-place outliers (quantizer.cu:83-104, 147-168): u32 codes, valid ones
// zigzag(q) in [0, 2 radius), an outlier's code is the raw bits of x; the
// inverse takes (code >> 1) >= radius as an outlier.
//
// Bitpack (modules/coders/bitpack/bitpack_stage.cu:30-124): the low `nbits`
// bits of each element, nbits in {1,2,4,8,16,32}; sub-byte: element k of a
// byte at bit k*nbits; multi-byte: little endian.
#include "fzh_compact.h"

namespace fzh {
namespace {

template <typename TCode> struct SignedOf;
template <> struct SignedOf<uint8_t> { using type = int8_t; };
template <> struct SignedOf<uint16_t> { using type = int16_t; };
template <> struct SignedOf<uint32_t> { using type = int32_t; };

// __float2int_rn: nearest-even; out of range saturates; NaN -> 0.
__device__ __forceinline__ int f2i_rn(float f) {
    if (f != f) return 0;
    if (f >= 2147483647.0f) return 2147483647;
    if (f <= -2147483648.0f) return (int)0x80000000;
    return (int)__builtin_rintf(f);
}

constexpr int QTILE = 1024;  // elements per wave (16 per lane)

template <typename TCode, bool ZZ>
__global__ void __launch_bounds__(256)
quant_fwd_kernel(const float* __restrict__ in, uint64_t n, float r, float threshold, int rad,
                 TCode* __restrict__ codes, float* __restrict__ sval, uint32_t* __restrict__ sidx,
                 uint32_t* __restrict__ scnt, uint32_t T) {
    using SC = typename SignedOf<TCode>::type;
    constexpr int W = 8 * sizeof(TCode);
    const uint32_t tile = blockIdx.x * 4 + wave_in_wg();
    if (tile < T) {
        const int l = lane_id();
        const uint64_t base = (uint64_t)tile * QTILE;
        float x[16];
        uint32_t mask = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint64_t e0 = base + 4 * (uint64_t)(l + 64 * q);
            if (e0 + 4 <= n) {
                const float4 v = *reinterpret_cast<const float4*>(in + e0);
                x[4 * q] = v.x; x[4 * q + 1] = v.y; x[4 * q + 2] = v.z; x[4 * q + 3] = v.w;
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) x[4 * q + k] = (e0 + k < n) ? in[e0 + k] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint64_t e = e0 + k;
                const int qv = f2i_rn(x[4 * q + k] * r);
                const bool ok = qv > -rad && qv < rad && fabsf(x[4 * q + k]) < threshold;
                TCode c = 0;
                if (ok) {
                    if constexpr (ZZ) {
                        const SC s = (SC)qv;
                        c = (TCode)(((TCode)s << 1) ^ (TCode)(s >> (W - 1)));
                    } else {
                        c = (TCode)qv;
                    }
                }
                if (e < n) {
                    codes[e] = c;
                    if (!ok) mask |= 1u << (4 * q + k);
                }
            }
        }
        const uint32_t agg = wave_sum(__popc(mask));
        if (agg) {
            uint32_t run = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t mq = (mask >> (4 * q)) & 0xFu;
                const uint32_t c = __popc(mq);
                const uint32_t incl = wave_incl_scan(c);
                uint32_t pos = run + incl - c;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (mq & (1u << k)) {
                        sval[base + pos] = x[4 * q + k];
                        sidx[base + pos] = (uint32_t)(base + 4 * (uint64_t)(l + 64 * q) + k);
                        pos++;
                    }
                run += lane63(incl);
            }
        }
        if (l == 0) scnt[tile] = agg;
    }
}

template <typename TCode, bool ZZ>
__global__ void __launch_bounds__(256)
quant_inv_kernel(const TCode* __restrict__ codes, uint64_t n, float ebx2, float* __restrict__ out) {
    using SC = typename SignedOf<TCode>::type;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const TCode c = codes[i];
        int q;
        if constexpr (ZZ) q = (int)(SC)((TCode)(c >> 1) ^ (TCode)(-(SC)(c & 1u)));
        else q = (int)(SC)c;
        out[i] = (float)q * ebx2;
    }
}

// ---------------------------------------------------------------------------
// REL: log2-space bins (quantizer.cu:171-352).  For x normal, finite and
// below the threshold: log_bin = __float2int_rn(log2|x| * log2eb_r), the
// code packs (|log_bin|, sign of log_bin, sign of x) + 1 (0 marks an
// outlier), and it is kept when |log_bin| < radius, it fits TCode and
// 2^(log_bin * log2eb) lies in [|x| / (1+eps), |x| (1+eps)]; everything else
// is an outlier.  The reference takes log2 and 2^t from __log2f / exp2f
// (within 2 ulp); here both are the correctly rounded float results (the
// double-precision functions rounded once), which is what the bin and the
// bound test are defined on.
// ---------------------------------------------------------------------------
struct RelParams {
    float log2eb, log2eb_r, opp, oopp;
};

__device__ __forceinline__ float log2_cr(float x) { return (float)log2((double)x); }
__device__ __forceinline__ float exp2_cr(float t) { return (float)exp2((double)t); }

// Code of one element (0: outlier).
template <typename TCode>
__device__ __forceinline__ uint32_t rel_code(float x, const RelParams& p, float threshold, uint32_t rad) {
    const uint32_t bits = __float_as_uint(x);
    const uint32_t expo = (bits >> 23) & 0xFFu;
    if (fabsf(x) >= threshold || expo == 0u || expo == 255u) return 0u;
    const bool neg = x < 0.0f;
    const float ax = neg ? -x : x;
    const int lb = f2i_rn(log2_cr(ax) * p.log2eb_r);
    const uint32_t alb = lb < 0 ? 0u - (uint32_t)lb : (uint32_t)lb;
    const uint32_t stored = ((alb << 2) | ((lb < 0 ? 1u : 0u) << 1) | (neg ? 1u : 0u)) + 1u;
    constexpr uint32_t cmax = sizeof(TCode) == 1 ? 0xFFu : sizeof(TCode) == 2 ? 0xFFFFu : 0xFFFFFFFFu;
    if (!(alb < rad && stored <= cmax)) return 0u;
    const float rec = exp2_cr((float)lb * p.log2eb);
    return (rec >= ax * p.oopp && rec <= ax * p.opp) ? stored : 0u;
}

template <typename TCode>
__global__ void __launch_bounds__(256)
quant_rel_fwd_kernel(const float* __restrict__ in, uint64_t n, RelParams p, float threshold, uint32_t rad,
                     TCode* __restrict__ codes, float* __restrict__ sval, uint32_t* __restrict__ sidx,
                     uint32_t* __restrict__ scnt, uint32_t T) {
    const uint32_t tile = blockIdx.x * 4 + wave_in_wg();
    if (tile >= T) return;
    const int l = lane_id();
    const uint64_t base = (uint64_t)tile * QTILE;
    float x[16];
    uint32_t mask = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint64_t e0 = base + 4 * (uint64_t)(l + 64 * q);
        if (e0 + 4 <= n) {
            const float4 v = *reinterpret_cast<const float4*>(in + e0);
            x[4 * q] = v.x; x[4 * q + 1] = v.y; x[4 * q + 2] = v.z; x[4 * q + 3] = v.w;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) x[4 * q + k] = (e0 + k < n) ? in[e0 + k] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint64_t e = e0 + k;
            const uint32_t c = rel_code<TCode>(x[4 * q + k], p, threshold, rad);
            if (e < n) {
                codes[e] = (TCode)c;
                if (c == 0u) mask |= 1u << (4 * q + k);
            }
        }
    }
    const uint32_t agg = wave_sum(__popc(mask));
    if (agg) {
        uint32_t run = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t mq = (mask >> (4 * q)) & 0xFu;
            const uint32_t c = __popc(mq);
            const uint32_t incl = wave_incl_scan(c);
            uint32_t pos = run + incl - c;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (mq & (1u << k)) {
                    sval[base + pos] = x[4 * q + k];
                    sidx[base + pos] = (uint32_t)(base + 4 * (uint64_t)(l + 64 * q) + k);
                    pos++;
                }
            run += lane63(incl);
        }
    }
    if (l == 0) scnt[tile] = agg;
}

// Inverse (quantizer.cu:328-352): code 0 -> 0 (an outlier's value is
// assigned afterwards), else +-2^(log_bin * log2eb).
template <typename TCode>
__global__ void __launch_bounds__(256)
quant_rel_inv_kernel(const TCode* __restrict__ codes, uint64_t n, float log2eb, float* __restrict__ out) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t st = (uint32_t)codes[i];
        float v = 0.0f;
        if (st != 0u) {
            const uint32_t cv = st - 1u;
            const int alb = (int)(cv >> 2);
            const int lb = ((cv >> 1) & 1u) ? -alb : alb;
            const float rec = exp2_cr((float)lb * log2eb);
            v = (cv & 1u) ? -rec : rec;
        }
        out[i] = v;
    }
}

// Grid-stride, one element per thread per step.
__global__ void __launch_bounds__(256)
quant_inplace_fwd_kernel(const float* __restrict__ in, uint64_t n, float r, float threshold, int rad,
                         uint32_t* __restrict__ codes) {
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
        const float x = in[i];
        const int q = f2i_rn(x * r);
        const bool ok = q > -rad && q < rad && fabsf(x) < threshold;
        codes[i] = ok ? (uint32_t)((q << 1) ^ (q >> 31)) : __float_as_uint(x);
    }
}

__global__ void __launch_bounds__(256)
quant_inplace_inv_kernel(const uint32_t* __restrict__ codes, uint64_t n, float ebx2, uint32_t rad,
                         float* __restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
        const uint32_t c = codes[i];
        if ((c >> 1) >= rad) {
            out[i] = __uint_as_float(c);
        } else {
            const int ci = (int)c;
            const int q = (ci & 1) ? -((ci + 1) >> 1) : (ci >> 1);
            out[i] = (float)q * ebx2;
        }
    }
}

__global__ void __launch_bounds__(256)
scatter_assign_kernel(const float* __restrict__ val, const uint32_t* __restrict__ idx,
                      const uint32_t* __restrict__ count, uint64_t max_out, uint64_t n, float* __restrict__ out) {
    const uint64_t k = min((uint64_t)*count, max_out);
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < k; t += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t i = idx[t];
        if (i < n) out[i] = val[t];
    }
}

// ---------------------------------------------------------------------------
// Bitpack
// ---------------------------------------------------------------------------
// Bound by memory: a thread takes 16 elements, which are whole 16-byte words
// of the elements and 2 * NB bytes of the packed array, so both sides move in
// wide accesses and the packing is constant shifts (6 Mi 16-bit codes at 16
// bits: 6.9 us; 10.5 with one byte store per output byte).  The last n % 16
// elements, at most 60 packed bytes, take a thread per byte.
template <int NB, typename F>
__device__ __forceinline__ void pack_tail(uint64_t n, uint8_t* __restrict__ out, uint64_t b0, uint64_t nout,
                                          uint32_t t, F&& element) {
    const uint64_t b = b0 + t;
    if (b >= nout) return;
    uint32_t v = 0;
    if constexpr (NB < 8) {
#pragma unroll
        for (int k = 0; k < 8 / NB; k++) {
            const uint64_t e = b * (8 / NB) + k;
            if (e < n) v |= (element(e) & ((1u << NB) - 1u)) << (k * NB);
        }
    } else {
        v = element(b / (NB / 8)) >> (8 * (b % (NB / 8)));
    }
    out[b] = (uint8_t)v;
}

template <typename T, int NB>
__global__ void __launch_bounds__(256)
bitpack_enc_vec_kernel(const T* __restrict__ in, uint64_t n, uint8_t* __restrict__ out) {
    constexpr uint32_t MASK = NB >= 32 ? 0xFFFFFFFFu : ((1u << (NB & 31)) - 1u);
    const uint64_t n16 = n / 16, stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n16; g += stride) {
        T v[16];
#pragma unroll
        for (int i = 0; i < (int)sizeof(T); i++)
            reinterpret_cast<uint4*>(v)[i] = reinterpret_cast<const uint4*>(in)[g * sizeof(T) + i];
        uint32_t o[(16 * NB + 31) / 32] = {};
#pragma unroll
        for (int e = 0; e < 16; e++) o[e * NB / 32] |= ((uint32_t)v[e] & MASK) << (e * NB % 32);
        uint8_t* d = out + g * 2 * NB;
        if constexpr (NB == 1) *reinterpret_cast<uint16_t*>(d) = (uint16_t)o[0];
        else if constexpr (NB == 2) *reinterpret_cast<uint32_t*>(d) = o[0];
        else if constexpr (NB == 4) *reinterpret_cast<uint2*>(d) = make_uint2(o[0], o[1]);
        else
#pragma unroll
            for (int i = 0; i < NB / 8; i++)
                reinterpret_cast<uint4*>(d)[i] = make_uint4(o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]);
    }
    if (blockIdx.x == 0)
        pack_tail<NB>(n, out, n16 * 2 * NB, (n * NB + 7) / 8, threadIdx.x, [&](uint64_t e) { return (uint32_t)in[e]; });
}

template <typename T, int NB>
__global__ void __launch_bounds__(256)
bitpack_dec_vec_kernel(const uint8_t* __restrict__ in, uint64_t n, T* __restrict__ out) {
    constexpr uint32_t MASK = NB >= 32 ? 0xFFFFFFFFu : ((1u << (NB & 31)) - 1u);
    const uint64_t n16 = n / 16, stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n16; g += stride) {
        const uint8_t* d = in + g * 2 * NB;
        uint32_t o[NB < 8 ? 2 : NB / 2];
        if constexpr (NB == 1) o[0] = *reinterpret_cast<const uint16_t*>(d);
        else if constexpr (NB == 2) o[0] = *reinterpret_cast<const uint32_t*>(d);
        else if constexpr (NB == 4) *reinterpret_cast<uint2*>(o) = *reinterpret_cast<const uint2*>(d);
        else
#pragma unroll
            for (int i = 0; i < NB / 8; i++) reinterpret_cast<uint4*>(o)[i] = reinterpret_cast<const uint4*>(d)[i];
        T v[16];
#pragma unroll
        for (int e = 0; e < 16; e++) v[e] = (T)((o[e * NB / 32] >> (e * NB % 32)) & MASK);
#pragma unroll
        for (int i = 0; i < (int)sizeof(T); i++)
            reinterpret_cast<uint4*>(out)[g * sizeof(T) + i] = reinterpret_cast<const uint4*>(v)[i];
    }
    const uint64_t e = n16 * 16 + threadIdx.x;
    if (blockIdx.x == 0 && e < n) {
        uint32_t v = 0;
        if constexpr (NB < 8) v = (in[e / (8 / NB)] >> ((e % (8 / NB)) * NB)) & MASK;
        else
#pragma unroll
            for (int b = 0; b < NB / 8; b++) v |= (uint32_t)in[e * (NB / 8) + b] << (8 * b);
        out[e] = (T)v;
    }
}

// One thread per packed byte (packing to less than 8 bits) or per element:
// arrays that are not 16-byte aligned (a thread per packed byte of wider
// elements loads each several times: 16 Mi 32-bit elements 67 us, 35), and
// unpacking of up to 16 bits to four-byte elements, where a group's 64 bytes per
// thread leave a wave's stores uncoalesced (16 Mi of 8 bits 24 us, 18 by elements;
// of 16 bits 25 and 26, but with the inverse that reads them 51 and 48 us for 6
// Mi; 32 bits 26 against 42).
template <typename T>
__global__ void __launch_bounds__(256)
bitpack_enc_kernel(const T* __restrict__ in, uint64_t n, int nbits, uint8_t* __restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (nbits < 8) {
        const uint64_t nout = (n * nbits + 7) / 8;
        const auto element = [&](uint64_t e) { return (uint32_t)in[e]; };
        for (uint64_t b = first; b < nout; b += stride) {
            switch (nbits) {
            case 1: pack_tail<1>(n, out, b, nout, 0, element); break;
            case 2: pack_tail<2>(n, out, b, nout, 0, element); break;
            default: pack_tail<4>(n, out, b, nout, 0, element); break;
            }
        }
    } else {
        const int bytes = nbits / 8;
        for (uint64_t i = first; i < n; i += stride) {
            uint32_t v = (uint32_t)in[i];
            for (int b = 0; b < bytes; b++) {
                out[i * bytes + b] = (uint8_t)v;
                v >>= 8;
            }
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
bitpack_dec_kernel(const uint8_t* __restrict__ in, uint64_t n, int nbits, T* __restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        if (nbits < 8) {
            const int epb = 8 / nbits;
            const uint32_t mask = (1u << nbits) - 1u;
            out[i] = (T)((in[i / epb] >> ((i % epb) * nbits)) & mask);
        } else {
            const int bytes = nbits / 8;
            uint32_t v = 0;
            for (int b = 0; b < bytes; b++) v |= (uint32_t)in[i * bytes + b] << (8 * b);
            out[i] = (T)v;
        }
    }
}

template <typename T, int NB>
void launch_bitpack_vec(hipStream_t s, bool enc, const void* in, size_t n, void* out) {
    if constexpr (NB <= 8 * (int)sizeof(T)) {
        const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(n / 16, 256), 8192));
        if (enc)
            bitpack_enc_vec_kernel<T, NB><<<blocks, 256, 0, s>>>((const T*)in, n, (uint8_t*)out);
        else if constexpr (sizeof(T) < 4 || NB > 16)
            bitpack_dec_vec_kernel<T, NB><<<blocks, 256, 0, s>>>((const uint8_t*)in, n, (T*)out);
    }
}

template <typename T>
void launch_bitpack(hipStream_t s, bool enc, const void* in, size_t n, int nbits, void* out) {
    const bool groups = enc || sizeof(T) < 4 || nbits > 16;
    if (groups && ((uintptr_t)in | (uintptr_t)out) % 16 == 0) {
        switch (nbits) {
        case 1: return launch_bitpack_vec<T, 1>(s, enc, in, n, out);
        case 2: return launch_bitpack_vec<T, 2>(s, enc, in, n, out);
        case 4: return launch_bitpack_vec<T, 4>(s, enc, in, n, out);
        case 8: return launch_bitpack_vec<T, 8>(s, enc, in, n, out);
        case 16: return launch_bitpack_vec<T, 16>(s, enc, in, n, out);
        default: return launch_bitpack_vec<T, 32>(s, enc, in, n, out);
        }
    }
    const size_t work = enc && nbits < 8 ? (n * nbits + 7) / 8 : n;
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(work, 256), 4096));
    if (enc)
        bitpack_enc_kernel<T><<<blocks, 256, 0, s>>>((const T*)in, n, nbits, (uint8_t*)out);
    else
        bitpack_dec_kernel<T><<<blocks, 256, 0, s>>>((const uint8_t*)in, n, nbits, (T*)out);
}

// Maximum in two launches: 16-byte loads, four in flight per thread, one
// partial maximum per workgroup, then one workgroup over the partials.  (One
// launch whose last workgroup finishes the reduction needs a device fence in
// every workgroup, which writes back the codes its XCD's L2 still holds: 26
// us for 6 Mi 2-byte codes, 131 with a single thread reading the partials;
// 5.9 us for the two launches.)  Up to MAX_ONE bytes one workgroup does it in one
// launch (3.4 us; 256 KiB that another launch has just written take it 9, though,
// where the two launches share their loads over many CUs).
constexpr size_t MAX_ONE = 32768;

template <typename T>
__device__ __forceinline__ void max_block(const T* __restrict__ in, uint64_t n, uint32_t* __restrict__ partial,
                                          uint32_t blk, uint32_t nblk) {
    __shared__ uint32_t sm[4];
    constexpr int E = 16 / sizeof(T);
    const uint64_t nv = (uintptr_t)in % 16 == 0 ? n / E : 0, stride = (uint64_t)nblk * blockDim.x;
    const uint64_t t = (uint64_t)blk * blockDim.x + threadIdx.x;
    uint32_t m = 0;
    for (uint64_t v0 = t; v0 < nv; v0 += 4 * stride) {
        uint4 w[4];
#pragma unroll
        for (int u = 0; u < 4; u++)
            w[u] = v0 + u * stride < nv ? reinterpret_cast<const uint4*>(in)[v0 + u * stride] : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int k = 0; k < E; k++) m = max(m, (uint32_t) reinterpret_cast<const T*>(&w[u])[k]);
    }
    for (uint64_t i = nv * E + t; i < n; i += stride) m = max(m, (uint32_t)in[i]);
    m = wave_max(m);
    if (lane_id() == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) partial[blk] = max(max(sm[0], sm[1]), max(sm[2], sm[3]));
}

template <typename T>
__global__ void __launch_bounds__(256)
max_partial_kernel(const T* __restrict__ in, uint64_t n, uint32_t* __restrict__ partial) {
    max_block<T>(in, n, partial, blockIdx.x, gridDim.x);
}

// Partial maxima together with the placement of the quantizer's or predictor's
// lists by the first `npl` workgroups: 6 Mi codes 4.8 us, 4.2 + 3.9 us and a gap
// as two launches.
template <typename T, int NL, typename V>
__global__ void __launch_bounds__(256)
max_partial_place_kernel(const T* __restrict__ in, uint64_t n, uint32_t* __restrict__ partial, CompactListT<V> L0,
                         CompactListT<V> L1, uint32_t PT, uint32_t PE, uint32_t npl) {
    if (blockIdx.x < npl) place_tiles<NL, true, V>(L0, L1, PT, PE, nullptr, blockIdx.x, npl);
    else max_block<T>(in, n, partial, blockIdx.x - npl, gridDim.x - npl);
}

__global__ void __launch_bounds__(256)
max_final_kernel(const uint32_t* __restrict__ partial, uint32_t np, uint32_t* __restrict__ result) {
    __shared__ uint32_t sm[4];
    uint32_t m = 0;
    for (uint32_t b = threadIdx.x; b < np; b += 256) m = max(m, partial[b]);
    m = wave_max(m);
    if (lane_id() == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) *result = max(max(sm[0], sm[1]), max(sm[2], sm[3]));
}

}  // namespace
}  // namespace fzh

namespace fzh {

int quant_abs_fwd_f32(hipStream_t s, const float* d_in, size_t n, float ebx2_r, float threshold, uint32_t radius,
                      int zigzag, int code_bytes, void* d_codes, float* d_oval, uint32_t* d_oidx, uint32_t* d_ocount,
                      size_t max_outliers, void* d_ws, size_t ws_bytes, PlaceDesc* defer) {
    if (ws_bytes < fzh_quant_abs_fwd_ws_bytes(n)) return fail(FZH_E_CAPACITY, "quantizer: workspace too small");
    if (n == 0) return FZH_OK;
    if (n > 0xFFFFFFFFull) return fail(FZH_E_INVALID, "quantizer: more than 2^32 elements");
    if ((uintptr_t)d_in % 16) return fail(FZH_E_INVALID, "quantizer: input must be 16-byte aligned");
    if (max_outliers > 0 && (!d_oval || !d_oidx)) return fail(FZH_E_INVALID, "quantizer: null outlier buffers");
    const uint32_t T = (uint32_t)cdiv(n, QTILE);
    const unsigned blocks = (unsigned)cdiv(T, 4);
    uint8_t* w = (uint8_t*)d_ws;
    const size_t o_cnt = compact_state_bytes(T);
    const size_t o_val = o_cnt + align_up(4 * (size_t)T, 256);
    const size_t o_idx = o_val + align_up(4 * (size_t)T * QTILE, 256);
    uint32_t* scnt = (uint32_t*)(w + o_cnt);
    float* sval = (float*)(w + o_val);
    uint32_t* sidx = (uint32_t*)(w + o_idx);
#define FZH_Q(TC, ZZV)                                                                                              \
    quant_fwd_kernel<TC, ZZV><<<blocks, 256, 0, s>>>(d_in, n, ebx2_r, threshold, (int)(TC)radius, (TC*)d_codes,   \
                                                     sval, sidx, scnt, T)
    switch (code_bytes) {
    case 1: if (zigzag) FZH_Q(uint8_t, true); else FZH_Q(uint8_t, false); break;
    case 2: if (zigzag) FZH_Q(uint16_t, true); else FZH_Q(uint16_t, false); break;
    case 4: if (zigzag) FZH_Q(uint32_t, true); else FZH_Q(uint32_t, false); break;
    default: return fail(FZH_E_INVALID, "quantizer: code_bytes must be 1, 2 or 4");
    }
#undef FZH_Q
    CompactList L0{sval, sidx, scnt, d_oval, d_oidx, d_ocount, max_outliers};
    FZH_CHECK_LAUNCH("quant_fwd_kernel");
    return launch_compact<float>(s, w, T, QTILE, L0, nullptr, defer);
}

int max_u32(hipStream_t s, const void* d_in, size_t n, int elem_bytes, uint32_t* d_max, void* d_ws, size_t ws_bytes,
            const PlaceDesc* place) {
    if (ws_bytes < fzh_max_u32_ws_bytes()) return fail(FZH_E_CAPACITY, "max: workspace too small");
    uint32_t* partial = (uint32_t*)((uint8_t*)d_ws + 256);
    const unsigned blocks = n * elem_bytes <= MAX_ONE ? 1u : (unsigned)std::min<size_t>(cdiv(n, 256 * 32), 1024);
    if (blocks == 1) partial = d_max;
    const auto launch = [&](auto tag) {
        using T = decltype(tag);
        if (place && place->blocks)
            with_placement(*place, [&](auto nl, auto L0, auto L1) {
                using V = std::remove_pointer_t<decltype(L0.val)>;
                max_partial_place_kernel<T, decltype(nl)::value, V><<<place->blocks + blocks, 256, 0, s>>>(
                    (const T*)d_in, n, partial, L0, L1, place->T, place->E, place->blocks);
            });
        else
            max_partial_kernel<T><<<blocks, 256, 0, s>>>((const T*)d_in, n, partial);
    };
    switch (elem_bytes) {
    case 1: launch(uint8_t{}); break;
    case 2: launch(uint16_t{}); break;
    case 4: launch(uint32_t{}); break;
    default: return fail(FZH_E_INVALID, "max: elem_bytes must be 1, 2 or 4");
    }
    if (blocks > 1) max_final_kernel<<<1, 256, 0, s>>>(partial, blocks, d_max);
    FZH_CHECK_LAUNCH("max_kernel");
    return FZH_OK;
}

}  // namespace fzh

using namespace fzh;

extern "C" {

// [compaction state][counts u32 x T][scratch values f32 x T*QTILE][scratch indices u32 x T*QTILE]
size_t fzh_quant_abs_fwd_ws_bytes(size_t n) {
    const size_t T = cdiv(std::max<size_t>(n, 1), QTILE);
    return compact_state_bytes(T) + align_up(4 * T, 256) + 2 * align_up(4 * T * QTILE, 256);
}

int fzh_quant_abs_fwd_f32(void* stream, const float* d_in, size_t n, float ebx2_r, float threshold, uint32_t radius,
                          int zigzag, int code_bytes, void* d_codes, float* d_oval, uint32_t* d_oidx,
                          uint32_t* d_ocount, size_t max_outliers, void* d_ws, size_t ws_bytes) {
    return quant_abs_fwd_f32(S(stream), d_in, n, ebx2_r, threshold, radius, zigzag, code_bytes, d_codes, d_oval, d_oidx,
                             d_ocount, max_outliers, d_ws, ws_bytes, nullptr);
}

int fzh_quant_abs_inv_f32(void* stream, const void* d_codes, size_t n, float ebx2, int zigzag, int code_bytes,
                          const float* d_oval, const uint32_t* d_oidx, const uint32_t* d_ocount, size_t max_outliers,
                          float* d_out) {
    if (n == 0) return FZH_OK;
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(n, 256), 4096));
    hipStream_t s = S(stream);
#define FZH_QI(TC, ZZV) quant_inv_kernel<TC, ZZV><<<blocks, 256, 0, s>>>((const TC*)d_codes, n, ebx2, d_out)
    switch (code_bytes) {
    case 1: if (zigzag) FZH_QI(uint8_t, true); else FZH_QI(uint8_t, false); break;
    case 2: if (zigzag) FZH_QI(uint16_t, true); else FZH_QI(uint16_t, false); break;
    case 4: if (zigzag) FZH_QI(uint32_t, true); else FZH_QI(uint32_t, false); break;
    default: return fail(FZH_E_INVALID, "quantizer: code_bytes must be 1, 2 or 4");
    }
#undef FZH_QI
    if (d_ocount && max_outliers > 0) {
        const unsigned ob = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(max_outliers, 256), 1024));
        scatter_assign_kernel<<<ob, 256, 0, s>>>(d_oval, d_oidx, d_ocount, max_outliers, n, d_out);
    }
    FZH_CHECK_LAUNCH("quantizer inverse");
    return FZH_OK;
}

void fzh_quant_rel_params(float eps, float* params) {
    const float log2eb = 2.0f * std::log2(1.0f + eps);  // quantizer.cu:563-568
    params[0] = log2eb;
    params[1] = 1.0f / log2eb;
    params[2] = 1.0f + eps;
    params[3] = 1.0f / (1.0f + eps);
}

int fzh_quant_rel_fwd_f32(void* stream, const float* d_in, size_t n, float eps, float threshold, uint32_t radius,
                          int code_bytes, void* d_codes, float* d_oval, uint32_t* d_oidx, uint32_t* d_ocount,
                          size_t max_outliers, void* d_ws, size_t ws_bytes) {
    if (ws_bytes < fzh_quant_abs_fwd_ws_bytes(n)) return fail(FZH_E_CAPACITY, "quantizer (REL): workspace too small");
    if (n == 0) return FZH_OK;
    if (n > 0xFFFFFFFFull) return fail(FZH_E_INVALID, "quantizer (REL): more than 2^32 elements");
    if (!d_in || !d_codes || !d_ocount) return fail(FZH_E_INVALID, "quantizer (REL): null pointer");
    if ((uintptr_t)d_in % 16) return fail(FZH_E_INVALID, "quantizer (REL): input must be 16-byte aligned");
    if (max_outliers > 0 && (!d_oval || !d_oidx)) return fail(FZH_E_INVALID, "quantizer (REL): null outlier buffers");
    float pf[4];
    fzh_quant_rel_params(eps, pf);
    const RelParams p{pf[0], pf[1], pf[2], pf[3]};
    const uint32_t T = (uint32_t)cdiv(n, QTILE);
    const unsigned blocks = (unsigned)cdiv(T, 4);
    uint8_t* w = (uint8_t*)d_ws;
    const size_t o_cnt = compact_state_bytes(T);
    const size_t o_val = o_cnt + align_up(4 * (size_t)T, 256);
    const size_t o_idx = o_val + align_up(4 * (size_t)T * QTILE, 256);
    uint32_t* scnt = (uint32_t*)(w + o_cnt);
    float* sval = (float*)(w + o_val);
    uint32_t* sidx = (uint32_t*)(w + o_idx);
    hipStream_t s = S(stream);
    switch (code_bytes) {
    case 1:
        launch_k("quant_rel_fwd_kernel", quant_rel_fwd_kernel<uint8_t>, dim3(blocks), dim3(256), 0, s, d_in, n, p,
                 threshold, (uint32_t)(uint8_t)radius, (uint8_t*)d_codes, sval, sidx, scnt, T);
        break;
    case 2:
        launch_k("quant_rel_fwd_kernel", quant_rel_fwd_kernel<uint16_t>, dim3(blocks), dim3(256), 0, s, d_in, n, p,
                 threshold, (uint32_t)(uint16_t)radius, (uint16_t*)d_codes, sval, sidx, scnt, T);
        break;
    case 4:
        launch_k("quant_rel_fwd_kernel", quant_rel_fwd_kernel<uint32_t>, dim3(blocks), dim3(256), 0, s, d_in, n, p,
                 threshold, radius, (uint32_t*)d_codes, sval, sidx, scnt, T);
        break;
    default: return fail(FZH_E_INVALID, "quantizer (REL): code_bytes must be 1, 2 or 4");
    }
    FZH_CHECK_LAUNCH("quant_rel_fwd_kernel");
    CompactList L0{sval, sidx, scnt, d_oval, d_oidx, d_ocount, max_outliers};
    return launch_compact<float>(s, w, T, QTILE, L0, nullptr);
}

int fzh_quant_rel_inv_f32(void* stream, const void* d_codes, size_t n, float eps, int code_bytes,
                          const float* d_oval, const uint32_t* d_oidx, const uint32_t* d_ocount, size_t max_outliers,
                          float* d_out) {
    if (n == 0) return FZH_OK;
    if (!d_codes || !d_out) return fail(FZH_E_INVALID, "quantizer (REL) inverse: null pointer");
    float pf[4];
    fzh_quant_rel_params(eps, pf);
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(n, 256), 4096));
    hipStream_t s = S(stream);
    switch (code_bytes) {
    case 1:
        launch_k("quant_rel_inv_kernel", quant_rel_inv_kernel<uint8_t>, dim3(blocks), dim3(256), 0, s,
                 (const uint8_t*)d_codes, n, pf[0], d_out);
        break;
    case 2:
        launch_k("quant_rel_inv_kernel", quant_rel_inv_kernel<uint16_t>, dim3(blocks), dim3(256), 0, s,
                 (const uint16_t*)d_codes, n, pf[0], d_out);
        break;
    case 4:
        launch_k("quant_rel_inv_kernel", quant_rel_inv_kernel<uint32_t>, dim3(blocks), dim3(256), 0, s,
                 (const uint32_t*)d_codes, n, pf[0], d_out);
        break;
    default: return fail(FZH_E_INVALID, "quantizer (REL): code_bytes must be 1, 2 or 4");
    }
    if (d_ocount && max_outliers > 0) {
        const unsigned ob = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(max_outliers, 256), 1024));
        launch_k("scatter_assign_kernel", scatter_assign_kernel, dim3(ob), dim3(256), 0, s, d_oval, d_oidx, d_ocount,
                 (uint64_t)max_outliers, (uint64_t)n, d_out);
    }
    FZH_CHECK_LAUNCH("quantizer (REL) inverse");
    return FZH_OK;
}

int fzh_quant_abs_fwd_inplace_f32(void* stream, const float* d_in, size_t n, float ebx2_r, float threshold,
                                  uint32_t radius, uint32_t* d_codes) {
    if (n == 0) return FZH_OK;
    if (!d_in || !d_codes) return fail(FZH_E_INVALID, "quantizer (in place): null pointer");
    if (radius == 0 || radius > (1u << 30)) return fail(FZH_E_INVALID, "quantizer (in place): radius must be in [1, 2^30]");
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(n, 256), 8192));
    quant_inplace_fwd_kernel<<<blocks, 256, 0, S(stream)>>>(d_in, n, ebx2_r, threshold, (int)radius, d_codes);
    FZH_CHECK_LAUNCH("quant_inplace_fwd_kernel");
    return FZH_OK;
}

int fzh_quant_abs_inv_inplace_f32(void* stream, const uint32_t* d_codes, size_t n, float ebx2, uint32_t radius,
                                  float* d_out) {
    if (n == 0) return FZH_OK;
    if (!d_codes || !d_out) return fail(FZH_E_INVALID, "quantizer (in place): null pointer");
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(n, 256), 8192));
    quant_inplace_inv_kernel<<<blocks, 256, 0, S(stream)>>>(d_codes, n, ebx2, radius, d_out);
    FZH_CHECK_LAUNCH("quant_inplace_inv_kernel");
    return FZH_OK;
}

size_t fzh_max_u32_ws_bytes(void) { return 256 + 4 * 1024; }

int fzh_max_u32(void* stream, const void* d_in, size_t n, int elem_bytes, uint32_t* d_max, void* d_ws,
                   size_t ws_bytes) {
    return max_u32(S(stream), d_in, n, elem_bytes, d_max, d_ws, ws_bytes, nullptr);
}

int fzh_bitpack_enc(void* stream, const void* d_in, size_t n, int elem_bytes, int nbits, void* d_out) {
    if (nbits <= 0 || nbits > 8 * elem_bytes || (nbits & (nbits - 1)) != 0)
        return fail(FZH_E_INVALID, "bitpack: nbits must be a power of two <= 8*sizeof(T)");
    if (n == 0) return FZH_OK;
    hipStream_t s = S(stream);
    switch (elem_bytes) {
    case 1: launch_bitpack<uint8_t>(s, true, d_in, n, nbits, d_out); break;
    case 2: launch_bitpack<uint16_t>(s, true, d_in, n, nbits, d_out); break;
    case 4: launch_bitpack<uint32_t>(s, true, d_in, n, nbits, d_out); break;
    default: return fail(FZH_E_INVALID, "bitpack: elem_bytes must be 1, 2 or 4");
    }
    FZH_CHECK_LAUNCH("bitpack_enc_kernel");
    return FZH_OK;
}

int fzh_bitpack_dec(void* stream, const void* d_in, size_t n, int elem_bytes, int nbits, void* d_out) {
    if (nbits <= 0 || nbits > 8 * elem_bytes || (nbits & (nbits - 1)) != 0)
        return fail(FZH_E_INVALID, "bitpack: nbits must be a power of two <= 8*sizeof(T)");
    if (n == 0) return FZH_OK;
    hipStream_t s = S(stream);
    switch (elem_bytes) {
    case 1: launch_bitpack<uint8_t>(s, false, d_in, n, nbits, d_out); break;
    case 2: launch_bitpack<uint16_t>(s, false, d_in, n, nbits, d_out); break;
    case 4: launch_bitpack<uint32_t>(s, false, d_in, n, nbits, d_out); break;
    default: return fail(FZH_E_INVALID, "bitpack: elem_bytes must be 1, 2 or 4");
    }
    FZH_CHECK_LAUNCH("bitpack_dec_kernel");
    return FZH_OK;
}

}  // extern "C"
