// huffman.hip — histogram and coarse Huffman encode/decode (gfx950).
//
// PHF stream (modules/coders/huffman/phf/hf_hl.cc:43-120, hf_buf.cc:151-176):
//   [phf_header 64 B][64 B (zeros here)][revbook][par_nbit u32 x pardeg]
//   [par_entry u32 x pardeg][bitstream u32 cells]
// phf_header: bklen (int:16) @0, sublen @4, pardeg @8, original_len u64 @16,
// total_nbit u64 @24, total_ncell u64 @32, entry[6] u32 @40 (entry[5] = total
// stream bytes).  Partitions of sublen = 768 symbols (coarse,
// hf_bk.cc:28-31) or 1024 (fine, the ReVISIT-lite path, hf_buf.cc:48-49);
// each partition's codewords are packed MSB-first into 32-bit cells
// (hf_kernels.cu:73-122, :145-250 build the same cells); par_entry =
// exclusive prefix of the per-partition cell counts.
//
// MI355X design
//   histogram: privatized per-wave LDS histograms, consecutive equal symbols
//     merged in-lane before the LDS atomic (the dominant code otherwise
//     serialises a 64-lane conflict).
//   encode: one wave per partition packs its codewords in parallel (a run of
//     symbols per lane, bit offsets from one wave prefix sum, whole cells
//     ORed into LDS) and writes them to the partition's scratch slot plus
//     par_nbit; a segmented device scan of the cell counts writes par_entry
//     into the stream; a pack kernel moves the cells (to a second destination
//     as well where there is one) and a one-workgroup kernel writes the
//     header: no host prefix sum, no host sync (reference phases 1-4 + two
//     syncs).
//   decode: a 2048-entry prefix table in LDS yields the symbol of any code
//     of up to 11 bits in one probe, chained tables those of longer ones.
//     Short streams: one wave per partition, 64 lanes decode equal spans of
//     its bits speculatively and settle the span starts in rounds (a prefix
//     code resynchronises within a few codewords); symbols are staged in LDS
//     and leave in 16-byte stores.  Long streams: one lane per partition
//     where their partitions, bits and runs make that the faster.
#include <type_traits>

#include "fzh_huffman_enc.h"
#include "fzh_scan.h"

namespace fzh {
namespace {

template <typename T>
__device__ __forceinline__ uint32_t ld_sym(const T* p, uint64_t i) { return (uint32_t)p[i]; }

// ---------------------------------------------------------------------------
// Histogram (histogram.cu:26-60 semantics: symbols >= bklen are skipped)
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
hist_kernel(const T* __restrict__ in, uint64_t n, uint32_t bklen, uint32_t* __restrict__ freq, int replicas) {
    extern __shared__ uint32_t sh[];
    const int wv = threadIdx.x >> 6;
    // 8 replicas: two per wave, by lane parity (half the same-bin lanes of
    // one LDS atomic); replica stride bklen + 1 words, so one bin of two
    // replicas sits in different banks
    const uint32_t rs = replicas == 8 ? bklen + 1 : bklen;
    const int rep = replicas == 8 ? 2 * wv + (threadIdx.x & 1) : (replicas == 4 ? wv : 0);
    for (uint32_t i = threadIdx.x; i < rs * (uint32_t)replicas; i += blockDim.x) sh[i] = 0;
    __syncthreads();
    uint32_t* h = sh + (size_t)rep * rs;
    constexpr int E = 16 / sizeof(T);
    const uint64_t nv = n / E;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    // four 16-byte loads per thread and step, issued before the atomics
    for (uint64_t v0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v0 < nv; v0 += 4 * stride) {
        uint4 w[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint64_t v = v0 + (uint64_t)u * stride;
            w[u] = v < nv ? reinterpret_cast<const uint4*>(in)[v] : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (v0 + (uint64_t)u * stride >= nv) continue;
            const T* p = reinterpret_cast<const T*>(&w[u]);
            uint32_t cur = (uint32_t)p[0], cnt = 1;
#pragma unroll
            for (int k = 1; k < E; k++) {
                const uint32_t s = (uint32_t)p[k];
                if (s == cur) {
                    cnt++;
                } else {
                    if (cur < bklen) atomicAdd(&h[cur], cnt);
                    cur = s;
                    cnt = 1;
                }
            }
            if (cur < bklen) atomicAdd(&h[cur], cnt);
        }
    }
    for (uint64_t i = nv * E + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint32_t s = (uint32_t)in[i];
        if (s < bklen) atomicAdd(&h[s], 1u);
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < bklen; b += blockDim.x) {
        uint32_t s = 0;
        for (int r = 0; r < replicas; r++) s += sh[(size_t)r * rs + b];
        if (s) atomicAdd(&freq[b], s);
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
hist_global_kernel(const T* __restrict__ in, uint64_t n, uint32_t bklen, uint32_t* __restrict__ freq) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t s = (uint32_t)in[i];
        if (s < bklen) atomicAdd(&freq[s], 1u);
    }
}

// ---------------------------------------------------------------------------
// Encode
// ---------------------------------------------------------------------------
constexpr unsigned ENC_BLOCKS = 4096;  // encode workgroups, at most

// Each workgroup stages the codebook once (bklen <= 8192: BOOK_LDS) and takes
// several partitions, one per wave at a time (huf_encode_partition); more
// workgroups (one partition a wave: 117 us for 2^27 symbols, now 96) stage it
// more often, fewer (2048: 103) leave too few waves to cover the loads.  A
// larger book stays in memory, and every wave takes one partition (2^25
// symbols of 16384: 93 us, 97 with ENC_BLOCKS).
template <typename T, int SL, bool BOOK_LDS>
__global__ void __launch_bounds__(256)
huf_enc_kernel(const T* __restrict__ in, uint64_t n, uint32_t bklen, const uint32_t* __restrict__ bk4,
               const uint8_t* __restrict__ revbook, uint32_t rev_bytes, uint8_t* __restrict__ out,
               uint32_t* __restrict__ scells, uint32_t* __restrict__ ncell_out, uint32_t pardeg) {
    constexpr int CELLS = cells_of(SL);
    extern __shared__ uint32_t smem[];
    const int wv = threadIdx.x >> 6;
    uint32_t* cells = smem + wv * CELLS;
    uint32_t* s_bk = smem + 4 * CELLS;
    if constexpr (BOOK_LDS) {
        for (uint32_t i = threadIdx.x; i < bklen; i += blockDim.x) s_bk[i] = bk4[i];
        __syncthreads();
    }
    const uint32_t ent1 = HDR_BYTES, ent2 = ent1 + rev_bytes;
    const int l = lane_id();
    const bool wide = (uintptr_t)in % enc_load_bytes<T, SL>() == 0;
    for (uint32_t p = blockIdx.x * 4 + wv; p < pardeg; p += gridDim.x * 4) {
        const uint64_t s0 = (uint64_t)p * SL;
        const uint32_t cnt = (uint32_t)((n - s0) < (uint64_t)SL ? (n - s0) : SL);
        const uint32_t nbit = huf_encode_partition<T, SL, BOOK_LDS>(in + s0, cnt, wide, s_bk, bk4, bklen, cells);
        const uint32_t ncell = (nbit + 31) / 32;
        uint32_t* dst = scells + (uint64_t)p * CELLS;
        for (uint32_t i = l; i < ncell; i += 64) dst[i] = cells[i];
        if (l == 0) {
            reinterpret_cast<uint32_t*>(out + ent2)[p] = nbit;
            ncell_out[p] = ncell;
        }
        if (p == 0) {
            for (uint32_t i = l; i < rev_bytes; i += 64) out[ent1 + i] = revbook[i];
            for (uint32_t i = 64 + l; i < HDR_BYTES; i += 64) out[i] = 0;
        }
        wave_lds_sync();
    }
}

// Cells of partition p -> stream cell par_entry[p] (one wave per partition);
// each workgroup adds its partitions' bit counts to one of NBIT_SLOTS
// accumulators (one atomic per workgroup) for the header.  With `copy` the
// stream goes there as well, the cells and what earlier launches wrote before
// them: for 2^27 symbols 57 -> 81 us here, but the concat of the caller's
// buffer 63 -> 32 as it doesn't read the stream again.
constexpr uint32_t NBIT_SLOTS = 256;

__global__ void __launch_bounds__(256)
huf_pack_kernel(const uint32_t* __restrict__ scells, const uint32_t* __restrict__ ncell,
                uint8_t* __restrict__ out, uint8_t* __restrict__ copy, uint32_t ent1, uint32_t ent2, uint32_t ent3, uint32_t ent4, uint32_t pardeg,
                uint32_t cells, unsigned long long* __restrict__ nbit_acc) {
    __shared__ uint32_t s_nb[4];
    const int w = (int)wave_in_wg();
    const uint32_t p = blockIdx.x * 4 + w;
    const int l = lane_id();
    uint32_t nb = 0;
    if (p < pardeg) {
        const uint32_t e = reinterpret_cast<const uint32_t*>(out + ent3)[p];
        const uint32_t c = ncell[p];
        const uint32_t* src = scells + (uint64_t)p * cells;
        uint32_t* dst = reinterpret_cast<uint32_t*>(out + ent4) + e;
        uint32_t* cdst = copy ? reinterpret_cast<uint32_t*>(copy + ent4) + e : nullptr;
        // up to four loads in flight per lane before their stores
        for (uint32_t i = l; i < c; i += 256) {
            uint32_t v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = i + 64 * k < c ? src[i + 64 * k] : 0u;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (i + 64 * k < c) dst[i + 64 * k] = v[k];
            if (copy)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (i + 64 * k < c) cdst[i + 64 * k] = v[k];
        }
        nb = reinterpret_cast<const uint32_t*>(out + ent2)[p];
    }
    if (copy) {  // the reverse book, and the workgroup's bit counts and entries
        const uint32_t* src = reinterpret_cast<const uint32_t*>(out);
        uint32_t* dst = reinterpret_cast<uint32_t*>(copy);
        for (uint32_t i = ent1 / 4 + blockIdx.x * 256 + threadIdx.x; i < ent2 / 4; i += gridDim.x * 256) dst[i] = src[i];
        const uint32_t q = blockIdx.x * 4 + (threadIdx.x & 3), i = (threadIdx.x & 4 ? ent3 : ent2) / 4 + q;
        if (threadIdx.x < 8 && q < pardeg) dst[i] = src[i];
    }
    if (l == 0) s_nb[w] = nb;
    __syncthreads();
    if (threadIdx.x == 0)  // spread over NBIT_SLOTS words: one address serialises every atomic
        atomicAdd(nbit_acc + (blockIdx.x % NBIT_SLOTS), (unsigned long long)s_nb[0] + s_nb[1] + s_nb[2] + s_nb[3]);
}

// phf_header (hf.h:38-44) once every partition is placed; sums the bit
// total from the NBIT_SLOTS accumulators and clears them for the next call.
__global__ void __launch_bounds__(256)
huf_header_kernel(uint8_t* __restrict__ out, uint8_t* __restrict__ copy, uint64_t n, uint32_t bklen, uint32_t sublen, uint32_t ent1, uint32_t ent2,
                  uint32_t ent3, uint32_t ent4, uint32_t pardeg, const uint32_t* __restrict__ total_ncell,
                  uint64_t* __restrict__ out_size, unsigned long long* __restrict__ nbit_acc) {
    __shared__ unsigned long long s_w[4];
    unsigned long long a = 0;
    for (uint32_t i = threadIdx.x; i < NBIT_SLOTS; i += 256) {
        a += nbit_acc[i];
        nbit_acc[i] = 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
    if (lane_id() == 0) s_w[threadIdx.x >> 6] = a;
    __syncthreads();
    if (copy)
        for (uint32_t i = 64 + threadIdx.x; i < HDR_BYTES; i += 256) copy[i] = 0;
    if (threadIdx.x == 0) {
        const unsigned long long tnb = s_w[0] + s_w[1] + s_w[2] + s_w[3];
        const uint32_t tc = *total_ncell;
        const uint32_t ent5 = ent4 + 4 * tc;
        for (uint8_t* o : {out, copy}) {
            if (!o) continue;
            uint32_t* h32 = reinterpret_cast<uint32_t*>(o);
            h32[0] = bklen & 0xFFFFu;
            h32[1] = sublen;
            h32[2] = pardeg;
            h32[3] = 0;
            reinterpret_cast<uint64_t*>(o)[2] = n;
            reinterpret_cast<uint64_t*>(o)[3] = tnb;
            reinterpret_cast<uint64_t*>(o)[4] = tc;
            h32[10] = 0;
            h32[11] = ent1;
            h32[12] = ent2;
            h32[13] = ent3;
            h32[14] = ent4;
            h32[15] = ent5;
        }
        *out_size = ent5;
    }
}

// ---------------------------------------------------------------------------
// Decode
// ---------------------------------------------------------------------------
// One wave per partition.  Codeword boundaries inside a partition are only
// known by decoding from its first bit, so the wave cuts the partition's
// bits into 64 equal spans (of at least 32 bits, longer than any codeword)
// and decodes them speculatively, all lanes at once: lane j starts at the
// first bit of span j and decodes the codewords that start inside its span,
// which leaves it at the end of its last codeword -- the first codeword
// boundary at or past span j+1's first bit, i.e. where lane j+1 really
// starts.  Lanes whose start moves decode again from the corrected start,
// and stop as soon as they reach a boundary of their previous decode (the
// first 64 bits of each span keep a boundary mask): from there on both
// decodes see the same codewords, so the count follows from the mask and
// the end is unchanged.  A prefix code falls back into step within a few
// codewords, so one short round nearly always settles the wave; lane 0 is
// always right and a lane whose predecessor is right becomes right in the
// next round, so 64 rounds bound it.  A prefix sum of the per-lane counts
// gives each lane its output offset; a last decode of each span writes its
// symbols to LDS and the wave stores the partition with 16-byte stores.
//
// Per codeword: a probe of a 2^11-entry table (length and symbol -- the
// symbol itself for 1- and 2-byte keys -- of every code of up to 11 bits);
// the prefixes of longer codes point into a second table indexed by as many
// more bits as fit, its long prefixes into a third, and so on (all codes
// that occur in typical books); codes longer still take the canonical
// comparison against the per-length limits first[l] << (32 - l), which do
// not increase with l (first[l] = round((first[l+1] + numl[l+1]) / 2)), so
// the length is one more than the number of limits above the window (the
// bit loop of hf_kernels.cu:258-312 in a few compares).  A window with no
// code of the book decodes as a 31-bit code with a flag that fails the
// partition, so the loops never branch on it.  Bits come from a 64-bit
// register buffer refilled from the partition's cells in LDS.
//
// A partition's cells are staged in LDS when they fit (DEC_CELLS cells and
// partitions of at most DEC_SUBLEN_MAX symbols, which covers the coarse 768
// and fine 1024 layouts); any other partition is decoded by the same steps
// reading its cells from memory and writing its symbols there.
constexpr int DEC_LUT_BITS = 11;
constexpr uint32_t DEC_LUT2 = 2048;     // entries of the second level, at most
constexpr uint32_t DEC_POOL = 3072;     // entries of the levels after the first
constexpr int DEC_LEVELS = 4;           // levels after the first
constexpr uint32_t DEC_CELLS = 448;
constexpr uint32_t DEC_SUBLEN_MAX = 1024;
constexpr uint32_t DEC_INVALID = 0xFFFFFFFFu;
// Table entry: value (symbol, or key index with DEC_KEY) in bits 0-23, code
// length in bits 24-28.  An entry with DEC_LONG is the prefix of longer
// codes and says where the next level's probe goes on: the window shifted
// left by bits 0-4, right by bits 5-9, plus the row's word offset in bits
// 10-23; DEC_DEEP where no level follows.
constexpr uint32_t DEC_KEY = 1u << 29;
constexpr uint32_t DEC_BAD = (1u << 30) | (31u << 24);  // no code: skip 31 bits, fail
constexpr uint32_t DEC_LONG = 1u << 31;
constexpr uint32_t DEC_DEEP = DEC_LONG | DEC_KEY;
constexpr uint32_t dec_probe(uint32_t row, uint32_t shl, uint32_t bits) { return (row << 10) | ((32 - bits) << 5) | shl; }
constexpr uint32_t DEC_LEVEL1 = dec_probe(0, 0, DEC_LUT_BITS);

// waves per workgroup: the tables are built once per workgroup, so
// workgroups are large; 4-byte keys halve it to keep the LDS under 64 KiB
template <typename T>
constexpr int dec_waves() { return sizeof(T) == 4 ? 4 : 8; }

struct DecTables {
    const uint32_t* lut;   // the levels one after another
    const uint64_t* lim;   // first[l] << (32 - l)
    const int32_t* diff;   // entry[l] - first[l]
    uint32_t maxl, nkeys;
};

// The entry that the probe st (DEC_LEVEL1 or a DEC_LONG entry) finds at W.
__device__ __forceinline__ uint32_t dec_lookup(const DecTables& t, uint32_t W, uint32_t st) {
    return t.lut[((st >> 10) & 0x3FFFu) + ((W << (st & 31u)) >> ((st >> 5) & 31u))];
}

// Entry of the code at the head of W, longer than every table level holds.
__device__ __forceinline__ uint32_t dec_deep(const DecTables& t, uint32_t W) {
    uint32_t lv = DEC_LUT_BITS + 1;
    for (uint32_t l = DEC_LUT_BITS + 1; l < t.maxl; l++) lv += (uint64_t)W < t.lim[l] ? 1u : 0u;
    const uint32_t k = (W >> (32 - lv)) + (uint32_t)t.diff[lv];
    if (lv > t.maxl || (uint64_t)W < t.lim[lv] || k >= t.nkeys) return DEC_BAD;
    return (lv << 24) | DEC_KEY | k;
}

// Entry of a code longer than DEC_LUT_BITS bits at the head of W, given its
// first-level entry e.
__device__ __forceinline__ uint32_t dec_long(const DecTables& t, uint32_t W, uint32_t e) {
    if (e < DEC_DEEP) {
        e = dec_lookup(t, W, e);
        if ((int32_t)e >= 0) return e;
        while (e < DEC_DEEP) {  // rows name later levels only
            e = dec_lookup(t, W, e);
            if ((int32_t)e >= 0) return e;
        }
    }
    return dec_deep(t, W);
}

__device__ __forceinline__ uint32_t dec_entry(const DecTables& t, uint32_t W) {
    uint32_t e = t.lut[W >> (32 - DEC_LUT_BITS)];
    if ((int32_t)e < 0) e = dec_long(t, W, e);
    return e;
}

// MSB-first reader of a partition's cells: staged in LDS (with zero cells
// past the end) or read from memory with the end checked.  `buf` holds bits
// [p, 32 next) of the partition at its top; it is refilled whenever fewer
// than 32 remain, i.e. when p > thr = 32 (next - 1).
template <bool STAGED>
struct DecBits {
    const uint32_t* c;
    uint32_t ncell;
    uint64_t buf;
    uint32_t next, thr;
    __device__ __forceinline__ uint32_t at(uint32_t k) const { return STAGED ? c[k] : (k < ncell ? c[k] : 0u); }
    __device__ __forceinline__ void seek(uint32_t p) {
        const uint32_t k = p >> 5;
        buf = (((uint64_t)at(k) << 32) | at(k + 1)) << (p & 31u);
        next = k + 2;
        thr = 32 * k + 32;
    }
    __device__ __forceinline__ uint32_t window() const { return (uint32_t)(buf >> 32); }
    // advance from p to p + L (L < 32)
    __device__ __forceinline__ void consume(uint32_t p, uint32_t L) {
        buf <<= L;
        p += L;
        if (p > thr) {
            buf |= (uint64_t)at(next) << (p - thr);
            next++;
            thr += 32;
        }
    }
};

// One partition of nbit bits and cnt symbols, decoded by one wave into
// `ost` (LDS staging, STAGED) or straight into `dst`.  Returns false if the
// bits do not decode to exactly cnt symbols ending at bit nbit.
template <typename T, bool STAGED>
__device__ __forceinline__ bool dec_partition(const uint32_t* cells, uint32_t ncell, const DecTables& t, uint32_t nbit,
                                              uint32_t cnt, const T* __restrict__ keys, T* ost, T* __restrict__ dst) {
    const uint32_t l = (uint32_t)lane_id();
    // spans of at least 32 bits: longer than any codeword, so every span
    // holds the start of a codeword and a correction moves on by whole spans
    const uint32_t seg = max((nbit + 63) / 64, 32u);
    const uint32_t act = (nbit + seg - 1) / seg;  // lanes with a span (wave-uniform, <= 64)
    if (act == 0) return cnt == 0;
    const bool on = l < act;
    const uint32_t lo = min(l * seg, nbit), lim = min(l * seg + seg, nbit);
    const uint32_t lim64 = min(lim, lo + 64);
    DecBits<STAGED> bits{cells, ncell, 0, 0, 0};
    // speculative decode from lo: count, end, boundaries in [lo, lo + 64)
    uint32_t b = lo, c = 0, e = nbit;
    uint64_t m = 0;
    if (on) {
        uint32_t p = lo, acc = 0;
        bits.seek(p);
        while (p < lim64) {
            const uint32_t en = dec_entry(t, bits.window());
            const uint32_t L = (en >> 24) & 31u;
            acc |= en;
            m |= 1ull << (p - lo);
            bits.consume(p, L);
            p += L;
            c++;
        }
        while (p < lim) {
            const uint32_t en = dec_entry(t, bits.window());
            const uint32_t L = (en >> 24) & 31u;
            acc |= en;
            bits.consume(p, L);
            p += L;
            c++;
        }
        e = (acc & (1u << 30)) ? DEC_INVALID : p;
    }
    for (int round = 0; round < 64; round++) {
        const uint32_t prev = wave_shr1(e);  // every lane takes part in the lane shift
        const uint32_t nb = l == 0 ? 0u : prev;
        const bool moved = on && nb != b;
        if (!__ballot(moved)) break;
        if (moved) {
            // decode again from nb, up to the first boundary of the previous decode
            b = nb;
            uint32_t p = nb, steps = 0, acc = 0;
            uint64_t mn = 0;
            bool synced = false;
            if (nb != DEC_INVALID) {
                bits.seek(p);
                while (p < lim64) {
                    if ((m >> (p - lo)) & 1ull) {
                        synced = true;
                        break;
                    }
                    const uint32_t en = dec_entry(t, bits.window());
                    const uint32_t L = (en >> 24) & 31u;
                    acc |= en;
                    mn |= 1ull << (p - lo);
                    bits.consume(p, L);
                    p += L;
                    steps++;
                }
            }
            if (nb == DEC_INVALID) {
                e = DEC_INVALID;
                c = 0;
                m = 0;
            } else if (synced && !(acc & (1u << 30))) {
                // from p on both decodes see the same codewords: e stays
                const uint64_t below = (1ull << (p - lo)) - 1ull;
                c = steps + c - (uint32_t)__popcll(m & below);
                m = mn | (m & ~below);
            } else {
                while (p < lim) {
                    const uint32_t en = dec_entry(t, bits.window());
                    const uint32_t L = (en >> 24) & 31u;
                    acc |= en;
                    bits.consume(p, L);
                    p += L;
                    steps++;
                }
                e = (acc & (1u << 30)) ? DEC_INVALID : p;
                c = steps;
                m = mn;
            }
        }
    }
    const uint32_t incl = wave_incl_scan(c);
    const uint32_t last_e = (uint32_t)__builtin_amdgcn_readlane((int)e, (int)(act - 1));
    if (last_e != nbit || lane63(incl) != cnt) return false;
    // every span settled: decode it once more, writing its symbols
    uint32_t o = incl - c;
    if (b < lim) {
        uint32_t p = b;
        bits.seek(p);
        while (p < lim) {
            const uint32_t en = dec_entry(t, bits.window());
            const uint32_t L = (en >> 24) & 31u;
            uint32_t v = en & 0xFFFFFFu;
            if (en & DEC_KEY) v = (uint32_t)keys[v];
            if (STAGED)
                ost[o] = (T)v;
            else
                dst[o] = (T)v;
            o++;
            bits.consume(p, L);
            p += L;
        }
    }
    return true;
}

// The stream's header fields, checked against n and the buffer size.
constexpr int cdiv_c(int a, int b) { return (a + b - 1) / b; }

struct DecHead {
    uint32_t sublen, pardeg, e1, nkeys, ncells;
    bool zero_len;  // a book of one symbol, whose code may have no bits
    const uint32_t* par_nbit;
    const uint32_t* par_entry;
    const uint32_t* cells;
};

template <typename T>
__device__ __forceinline__ bool dec_head(const uint8_t* __restrict__ in, uint64_t in_bytes, uint64_t n, DecHead& h) {
    if (in_bytes < HDR_BYTES) return false;
    const int32_t sublen = *reinterpret_cast<const int32_t*>(in + 4);
    const int32_t pardeg = *reinterpret_cast<const int32_t*>(in + 8);
    const uint32_t* ent = reinterpret_cast<const uint32_t*>(in + 40);
    const uint32_t e1 = ent[1], e2 = ent[2], e3 = ent[3], e4 = ent[4], e5 = ent[5];
    if (!(sublen > 0 && pardeg >= 0 && (uint64_t)pardeg == (n + sublen - 1) / sublen && e1 <= e2 && e2 - e1 >= 256 &&
          (e2 - e1 - 256) / sizeof(T) <= 65536 && e2 <= e3 && e3 <= e4 && e4 <= e5 && e5 <= in_bytes &&
          e3 - e2 == 4ull * pardeg && e4 - e3 == 4ull * pardeg && (e4 % 4) == 0 && (e1 % 4) == 0))
        return false;
    h.sublen = (uint32_t)sublen;
    h.pardeg = (uint32_t)pardeg;
    h.e1 = e1;
    h.nkeys = (e2 - e1 - 256) / sizeof(T);
    h.ncells = (e5 - e4) / 4;
    h.par_nbit = reinterpret_cast<const uint32_t*>(in + e2);
    h.par_entry = reinterpret_cast<const uint32_t*>(in + e3);
    h.cells = reinterpret_cast<const uint32_t*>(in + e4);
    h.zero_len = reinterpret_cast<const uint32_t*>(in + e1)[33] == 1;  // entry[1]
    return true;
}

struct DecLds {
    uint32_t lut[(1 << DEC_LUT_BITS) + DEC_POOL];
    uint64_t lim[32];
    int32_t diff[32];
};

// One table level: entry i (of `count`) stands for the window whose top
// bits are i in L0 + b bits; codes of (L0, L0 + b] bits get their entry,
// longer ones longer(i).  A code's length is the first l at which its top
// l bits reach first[l] (the bit loop of hf_kernels.cu:258-312); fv holds
// first[l] in lane l, so the compares are independent and their operands
// scalar, and a thread's keys are loaded together.
template <typename T, int BLOCK, int PER, typename F>
__device__ __forceinline__ void dec_level(uint32_t* tab, uint32_t count, uint32_t l0, uint32_t b, uint32_t fv,
                                          const int32_t* diff, const T* __restrict__ keys, uint32_t nkeys, F&& longer) {
    constexpr bool FOLD = sizeof(T) <= 2;
    // The trip count is the wave's (its first entry < count), so readlane never
    // names a lane that has left the loop, whose copy of fv no instruction need
    // keep; lanes past `count` compute an entry that they don't store.
    const uint32_t lane = (uint32_t)lane_id();
    for (uint32_t w0 = wave_in_wg() * 64; w0 < count; w0 += BLOCK * PER) {
        const uint32_t i0 = w0 + lane;
        uint32_t W[PER], lv[PER], k[PER], key[PER];
#pragma unroll
        for (int i = 0; i < PER; i++) {
            W[i] = (i0 + i * BLOCK) << (32 - l0 - b);
            lv[i] = 0;
        }
        for (uint32_t l = l0 + b; l > l0; l--) {
            const uint32_t f = (uint32_t)__builtin_amdgcn_readlane((int)fv, (int)l);
#pragma unroll
            for (int i = 0; i < PER; i++)
                if ((W[i] >> (32 - l)) >= f) lv[i] = l;
        }
#pragma unroll
        for (int i = 0; i < PER; i++) k[i] = lv[i] ? (W[i] >> (32 - lv[i])) + (uint32_t)diff[lv[i]] : 0u;
#pragma unroll
        for (int i = 0; i < PER; i++)
            key[i] = FOLD && lv[i] && k[i] < nkeys ? (uint32_t)keys[k[i]] : (DEC_KEY | k[i]);
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (i0 + i * BLOCK < count)
                tab[i0 + i * BLOCK] =
                    lv[i] == 0 ? longer(i0 + i * BLOCK) : (k[i] >= nkeys ? DEC_BAD : (lv[i] << 24) | key[i]);
    }
}

// Builds the tables of the stream's book (all BLOCK threads; ends with a
// barrier).
template <typename T, int BLOCK>
__device__ __forceinline__ DecTables dec_build(const uint8_t* __restrict__ in, const DecHead& h, DecLds& t) {
    const uint32_t* fb = reinterpret_cast<const uint32_t*>(in + h.e1);
    const T* keys = reinterpret_cast<const T*>(in + h.e1 + 256);
    const uint32_t nkeys = h.nkeys;
    // lane l < 32 of every wave: first[l], entry[l]; is l a code length of the book?
    const uint32_t l32 = (uint32_t)lane_id() & 31u;
    const uint32_t fv = fb[l32], en = fb[32 + l32], en1 = l32 < 31 ? fb[33 + l32] : nkeys;
    const uint32_t used = (uint32_t)__ballot(l32 > 0 && en1 > en);
    // the longest length a window can have: the last with a code, or the
    // first at which every value is one (first[l] = 0)
    const uint32_t all = (uint32_t)__ballot(l32 > 0 && fv == 0);
    uint32_t maxl = used ? 31u - (uint32_t)__builtin_clz(used) : 1u;
    if (all) maxl = min(maxl, (uint32_t)__builtin_ctz(all));
    if (threadIdx.x < 32) {
        t.lim[threadIdx.x] = threadIdx.x ? (uint64_t)fv << (32 - threadIdx.x) : ~0ull;
        t.diff[threadIdx.x] = (int32_t)(en - fv);
    }
    __syncthreads();
    // The long codes' prefixes are [0, first[l]) at every length l (the
    // smallest values of their lengths), so a level is indexed by the prefix
    // that is still long and as many more bits as fit its part of the pool.
    uint32_t lev_l[DEC_LEVELS], lev_b[DEC_LEVELS], lev_n[DEC_LEVELS], lev_o[DEC_LEVELS];
    uint32_t at = DEC_LUT_BITS, off = 1u << DEC_LUT_BITS;
#pragma unroll
    for (int j = 0; j < DEC_LEVELS; j++) {
        const uint32_t room = (1u << DEC_LUT_BITS) + DEC_POOL - off;
        const uint32_t cap = j == 0 ? DEC_LUT2 : room - room / 4;
        const uint32_t c = maxl > at ? (uint32_t)__builtin_amdgcn_readlane((int)fv, (int)at) : 0u;
        uint32_t b = 0;
        if (c > 0)
            while (b < maxl - at && ((uint64_t)c << (b + 1)) <= cap) b++;
        lev_l[j] = at;
        lev_b[j] = b;
        lev_n[j] = b ? c << b : 0u;
        lev_o[j] = off;
        off += lev_n[j];
        at += b;
    }
    const auto next = [&](int j, uint32_t i) {  // entry of a code longer than the level before level j
        return j < DEC_LEVELS && lev_b[j] ? DEC_LONG | dec_probe(lev_o[j] + (i << lev_b[j]), lev_l[j], lev_b[j])
                                          : DEC_DEEP;
    };
    dec_level<T, BLOCK, cdiv_c(1 << DEC_LUT_BITS, BLOCK)>(t.lut, 1u << DEC_LUT_BITS, 0, DEC_LUT_BITS, fv, t.diff, keys,
                                                          nkeys, [&](uint32_t i) { return next(0, i); });
#pragma unroll
    for (int j = 0; j < DEC_LEVELS; j++)
        if (lev_n[j])
            dec_level<T, BLOCK, 4>(t.lut + lev_o[j], lev_n[j], lev_l[j], lev_b[j], fv, t.diff, keys, nkeys,
                                   [&](uint32_t i) { return next(j + 1, i); });
    __syncthreads();
    return DecTables{t.lut, t.lim, t.diff, maxl, nkeys};
}

// A partition whose book has one symbol with a zero-length code.
template <typename T>
__device__ __forceinline__ void dec_constant(T* __restrict__ dst, uint32_t cnt, T v) {
    constexpr uint32_t E = 16 / sizeof(T);
    uint32_t done = 0;
    if (((uintptr_t)dst & 15u) == 0) {
        const uint32_t w = sizeof(T) == 4 ? (uint32_t)v : (uint32_t)v * (sizeof(T) == 1 ? 0x01010101u : 0x00010001u);
        for (uint32_t j = (uint32_t)lane_id(); j < cnt / E; j += 64) reinterpret_cast<uint4*>(dst)[j] = make_uint4(w, w, w, w);
        done = cnt / E * E;
    }
    for (uint32_t j = done + (uint32_t)lane_id(); j < cnt; j += 64) dst[j] = v;
}

// Partition p, decoded by one wave; cst and ost: the wave's DEC_CELLS + 4 words
// and DEC_SUBLEN_MAX symbols of LDS.
template <typename T>
__device__ __forceinline__ void dec_wave(const DecHead& h, const DecTables& tb, const T* __restrict__ keys,
                                         uint32_t p, uint64_t n, T* __restrict__ out, uint32_t* cst, uint4* ost,
                                         int* __restrict__ d_status) {
    const uint32_t l = (uint32_t)lane_id();
    const uint32_t nbit = h.par_nbit[p];
    const uint32_t pe = h.par_entry[p];
    const uint32_t ncell = (uint32_t)(((uint64_t)nbit + 31) / 32);
    const uint64_t o0 = (uint64_t)p * h.sublen;
    const uint32_t cnt = (uint32_t)((n - o0) < (uint64_t)h.sublen ? (n - o0) : (uint64_t)h.sublen);
    T* dst = out + o0;
    if ((uint64_t)pe + ncell > h.ncells) {
        if (l == 0) *d_status = 1;
        return;
    }
    if (h.zero_len && nbit == 0) {
        dec_constant(dst, cnt, h.nkeys ? keys[0] : (T)0);
        return;
    }
    bool ok;
    if (ncell <= DEC_CELLS && h.sublen <= DEC_SUBLEN_MAX) {
        wave_lds_sync();  // the previous partition's staging reads are done
        for (uint32_t i = l; i < ncell + 4; i += 64) cst[i] = i < ncell ? h.cells[pe + i] : 0u;
        wave_lds_sync();
        T* st = reinterpret_cast<T*>(ost);
        ok = dec_partition<T, true>(cst, ncell, tb, nbit, cnt, keys, st, dst);
        wave_lds_sync();
        if (ok) {
            const uint32_t bytes = cnt * (uint32_t)sizeof(T);
            uint32_t done = 0;
            if (((uintptr_t)dst & 15u) == 0) {
                const uint32_t nv = bytes / 16;
                for (uint32_t i = l; i < nv; i += 64) reinterpret_cast<uint4*>(dst)[i] = ost[i];
                done = nv * 16 / (uint32_t)sizeof(T);
            }
            for (uint32_t i = done + l; i < cnt; i += 64) dst[i] = st[i];
        }
    } else {
        ok = dec_partition<T, false>(h.cells + pe, ncell, tb, nbit, cnt, keys, nullptr, dst);
    }
    if (!ok && l == 0) *d_status = 1;
}

template <typename T>
__global__ void __launch_bounds__(64 * dec_waves<T>())
huf_dec_kernel(const uint8_t* __restrict__ in, uint64_t in_bytes, T* __restrict__ out, uint64_t n,
               int* __restrict__ d_status) {
    constexpr int DEC_WAVES = dec_waves<T>();
    __shared__ DecLds s_tab;
    __shared__ uint32_t s_cells[DEC_WAVES][DEC_CELLS + 4];
    __shared__ uint4 s_out[DEC_WAVES][DEC_SUBLEN_MAX * sizeof(T) / 16];
    DecHead h;
    if (!dec_head<T>(in, in_bytes, n, h)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *d_status = 1;
        return;
    }
    const T* keys = reinterpret_cast<const T*>(in + h.e1 + 256);
    const DecTables tb = dec_build<T, 64 * DEC_WAVES>(in, h, s_tab);
    const uint32_t w = wave_in_wg();
    for (uint32_t p = blockIdx.x * DEC_WAVES + w; p < h.pardeg; p += gridDim.x * DEC_WAVES)
        dec_wave<T>(h, tb, keys, p, n, out, s_cells[w], s_out[w], d_status);
}

// ---------------------------------------------------------------------------
// Decode, one lane per partition (long streams)
// ---------------------------------------------------------------------------
// A lane that owns a partition decodes it from its first bit: every codeword
// once, where the wave-per-partition kernel decodes each two to three times
// (speculative spans, corrections, the writing pass) and waits for the
// slowest of 64 lanes in each.  Every step is one table probe for all 64
// lanes; a lane whose probe names a longer code goes on in the next level
// with its next step instead of in a branch (2% of the codewords of a
// spiky field are long, which is some lane of the wave in 3 steps of 4: the
// branch took 160 instead of 113 us on a lone wave, and 670 where whole
// partitions hold the longest codes).  Lanes drift apart by their long codes
// and each writes its own place of the output.
//   bits in: the lane's next 8 cells are always in flight or held in
//     registers (two 16-byte loads) and go into its 16-cell LDS ring when 8
//     cells are free, which is checked once per 8 steps (they use at most 8
//     cells); the ring's 16-byte pieces are rotated by lane, so lanes at
//     equal positions use different banks.
//   symbols out: a strip of two 16-symbol segments per lane in LDS; every 16
//     steps the wave stores the segments that are full, 32 bytes of each of
//     its 64 partitions (2-byte symbols).
// Serial over a partition (about 113 us for 768 symbols on any stream), and
// bound by VALU issue (33 instructions a step) beside the LDS probe latency
// once three waves share a SIMD: 2^27 symbols 244 us, one wave per partition
// 595 / 490 (spiky / smooth field).  dec_by_lanes says which streams.
constexpr int DECL_WAVES = 4;  // with 52.4 KiB of LDS three workgroups fit a CU: three waves per SIMD

typedef uint32_t huf_u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

template <typename T>
struct LaneDec {
    uint32_t* ring;  // this lane's 16 cells, pieces rotated by rot
    uint32_t rot;    // 4 * (lane / 4 % 4)
    uint32_t base;   // the partition's first cell
    uint32_t left;   // cells from there to the end of the stream
    uint32_t F;      // cells [F, F + 8) are in q, [.., F) in the ring
    uint32_t rp;     // next cell to read from the ring
    uint4 q0, q1;
    uint32_t w0, w1, s;  // window = {w0, w1} >> s, s < 32; w1 = cell rp - 1

    // Both arms write whole tuples: with the tail's words loaded behind a branch
    // each, the compiler lost one word of a tuple (its store's address was
    // computed into the tuple's own second register).
    __device__ __forceinline__ void fetch(const DecHead& h) {
        // the stream is below 4 GiB: 32-bit byte offsets
        const char* c = reinterpret_cast<const char*>(h.cells);
        if (F + 8 <= left) {
            const uint32_t o = 4 * (base + F);
            const huf_u32x4_a4 x = *reinterpret_cast<const huf_u32x4_a4*>(c + o);
            const huf_u32x4_a4 y = *reinterpret_cast<const huf_u32x4_a4*>(c + o + 16);
            q0 = make_uint4(x.x, x.y, x.z, x.w);
            q1 = make_uint4(y.x, y.y, y.z, y.w);
        } else {  // the stream's last cells (it has one: dec_by_lanes), zeros past them
            uint32_t v[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) {
                const uint32_t k = min(base + min(F + i, left), h.ncells - 1);
                v[i] = *reinterpret_cast<const uint32_t*>(c + 4 * k);
            }
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) v[i] = F + i < left ? v[i] : 0u;
            q0 = make_uint4(v[0], v[1], v[2], v[3]);
            q1 = make_uint4(v[4], v[5], v[6], v[7]);
        }
    }
    __device__ __forceinline__ void commit() {
        *reinterpret_cast<uint4*>(ring + ((F + rot) & 15u)) = q0;
        *reinterpret_cast<uint4*>(ring + ((F + 4 + rot) & 15u)) = q1;
        F += 8;
    }
    // keeps at least 9 unread cells in the ring (a block reads at most 8)
    __device__ __forceinline__ void refill(const DecHead& h) {
        if (F - rp <= 8) {
            commit();
            fetch(h);
        }
    }
    __device__ __forceinline__ uint32_t peek() const { return ring[(rp + rot) & 15u]; }
    __device__ __forceinline__ void start(const DecHead& h, uint32_t pe) {
        base = pe;
        left = h.ncells - pe;  // pe <= ncells: checked by the caller
        F = rp = 0;
        fetch(h);
        commit();
        fetch(h);
        commit();
        fetch(h);
        w0 = 0;
        w1 = peek();
        rp = 1;
        s = 0;
    }
    __device__ __forceinline__ uint32_t window() const { return __builtin_amdgcn_alignbit(w0, w1, s); }
    // L < 32 bits on; nx = peek() from before the entry was known, so its
    // LDS read runs beside the table's (reading only in the lanes that need
    // it, after the table's, was 138 instead of 113 us on a lone wave)
    __device__ __forceinline__ void consume(uint32_t L, uint32_t nx) {
        const bool c = s < L;
        w0 = c ? w1 : w0;
        w1 = c ? nx : w1;
        rp += c ? 1u : 0u;
        s = (s - L) & 31u;
    }
    __device__ __forceinline__ uint32_t bitpos() const { return 32 * (rp - 1) - s; }
};

// The wave's 64 partitions from p0 (lanes past the last have no symbols).
template <typename T>
__device__ __forceinline__ void dec_lanes(const DecHead& h, const DecTables& t, const T* __restrict__ keys,
                                          uint32_t p0, uint64_t n, T* __restrict__ out, uint32_t* ring,
                                          uint32_t* strip, int* __restrict__ d_status) {
    constexpr uint32_t SEG = 16;                            // symbols per stored segment
    constexpr uint32_t SW = 2 * SEG * sizeof(T) / 4;        // words of a lane's strip (two segments)
    constexpr uint32_t PIECES = SEG * sizeof(T) / 16;       // 16-byte pieces of a segment
    const uint32_t l = (uint32_t)lane_id();
    const uint32_t p = p0 + l;
    const bool on = p < h.pardeg;
    const uint64_t o0 = (uint64_t)p * h.sublen;
    const uint32_t cnt = !on ? 0u : (uint32_t)((n - o0) < (uint64_t)h.sublen ? (n - o0) : (uint64_t)h.sublen);
    const uint32_t nbit = on ? h.par_nbit[p] : 0u;
    LaneDec<T> d;
    d.ring = ring + 16 * l;
    d.rot = l & 12u;
    d.start(h, on ? h.par_entry[p] : 0u);
    // symbol k of the lane at byte (k sizeof(T) + 4 (l / 4)) mod strip size
    T* my = reinterpret_cast<T*>(strip + SW * l);
    constexpr uint32_t MASK = 2 * SEG - 1;
    const uint32_t turn = (l >> 2) * (4 / (uint32_t)sizeof(T));
    const uint32_t end = turn + cnt;
    uint32_t k = turn, flushed = 0;  // turn + symbols decoded, segments stored
    uint32_t st = DEC_LEVEL1, acc = 0;
    while (__ballot(k < end)) {
        for (int blk = 0; blk < 2; blk++) {
            d.refill(h);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t nx = d.peek();
                const uint32_t W = d.window();
                uint32_t e = dec_lookup(t, W, st);
                if (e >= DEC_DEEP) {
                    e = dec_deep(t, W);
                    if (e & DEC_KEY) e = (e & (31u << 24)) | (uint32_t)keys[e & 0xFFFFFFu];
                }
                const bool more = (int32_t)e < 0;
                my[k & MASK] = (T)e;  // past the lane's last symbol: a free slot
                const bool emit = !more && k < end;
                const uint32_t em = emit ? e : 0u;
                acc |= em;
                k += emit ? 1u : 0u;
                st = more ? e : DEC_LEVEL1;
                d.consume((em >> 24) & 31u, nx);
            }
        }
        // 16 probes decode at most 16 symbols, so after this at most 15 wait
        wave_lds_sync();
        const uint32_t mine = (flushed << 1) | (k - turn >= SEG * (flushed + 1) ? 1u : 0u);
#pragma unroll
        for (uint32_t i = 0; i < PIECES; i++) {
            const uint32_t r = (64 / PIECES) * i + l / PIECES, c = l % PIECES;
            const uint32_t v = (uint32_t)__shfl((int)mine, (int)r, 64);
            const uint32_t f = v >> 1;
            const uint32_t* row = strip + SW * r;
            const uint32_t w0 = (f & 1u) * (SW / 2) + 4 * c + (r >> 2);
            const uint4 x = make_uint4(row[w0 & (SW - 1)], row[(w0 + 1) & (SW - 1)], row[(w0 + 2) & (SW - 1)],
                                       row[(w0 + 3) & (SW - 1)]);
            if (v & 1u) gst_u4(out + (uint64_t)(p0 + r) * h.sublen + f * SEG + c * (16 / (uint32_t)sizeof(T)), x);
        }
        flushed += mine & 1u;
        wave_lds_sync();
    }
    for (uint32_t j = SEG * flushed; j < k - turn; j++) out[o0 + j] = my[(j + turn) & MASK];  // the last partition's remainder
    if (on && ((acc & (1u << 30)) || d.bitpos() != nbit)) *d_status = 1;
}

// Streams of at least this many coarse partitions are decoded by lanes or by
// waves as dec_by_lanes says; shorter ones by waves.
constexpr size_t DECL_MIN_PARTS = 32768;
constexpr unsigned DEC_MAX_BLOCKS = 768;  // of the decode by waves: three per CU

// What the two take, from 24 Mi to 48 Mi symbols of 1.1 to 7.7 bits:
//   lanes  0.168 us (2-byte keys; 1-byte 0.156) a symbol of a partition, for
//          any number of partitions up to a wave per SIMD (65536)
//   waves  a partition: 1.35 ns, 0.4 (0.35) a bit of its average code, 0.06 for
//          each codeword that a lane's span of at least 32 bits holds beyond
//          a 64th of the partition; 10 more where it repeats one code of two
//          or more bits, as spans then never fall into step and settle one lane
//          a round
// Waves / lanes in us, partitions of 768 symbols, 2-byte keys, bits a symbol in
// brackets: 24 Mi symbols [7.3] 145 / 126, [2.8] 82 / 128, [1.1] 87 / 109; 36 Mi
// 214 / 128, 118 / 130, 131 / 111; 48 Mi 264 / 130, 141 / 131, 165 / 112; 32 Mi in
// runs 560 / 107.  1024 symbols [7.3]: 24 Mi 117 / 173, 36 Mi 169 / 175, 48 Mi
// 215 / 176.  Partitions of more than DEC_SUBLEN_MAX symbols (the encoder writes 768
// and 1024), or whose segments of 16 are not 16-byte aligned, go by waves.
template <typename T>
__device__ __forceinline__ bool dec_by_lanes(const DecHead& h, uint64_t n) {
    if (h.sublen % 16 != 0 || h.sublen > DEC_SUBLEN_MAX || h.zero_len || h.ncells == 0) return false;
    constexpr float LANE = sizeof(T) == 1 ? 156.0f : 168.0f, BIT = sizeof(T) == 1 ? 0.35f : 0.4f;  // ns
    const float lanes = LANE * (float)h.sublen;
    const float bits = 32.0f * (float)h.ncells / (float)n;
    const float steps = 32.0f / bits - (float)h.sublen / 64.0f;
    const float wave = 1.35f + BIT * bits + (steps > 0.0f ? 0.06f * steps : 0.0f);
    if (wave * (float)h.pardeg > lanes) return true;
    // two cells in the middle of 64 partitions across the stream: do they
    // repeat with a period of up to 12 bits?
    const uint32_t p = (uint32_t)((uint64_t)lane_id() * (h.pardeg - 1) / 64);
    const uint32_t nbit = h.par_nbit[p], at = h.par_entry[p] + nbit / 64;
    bool repeats = false;
    if (nbit >= h.sublen + h.sublen / 2 && (uint64_t)at + 2 <= h.ncells) {
        const uint64_t w = ((uint64_t)h.cells[at] << 32) | h.cells[at + 1];
#pragma unroll
        for (int l = 1; l <= 12; l++) repeats |= ((w ^ (w << l)) >> l) == 0;
    }
    const float runs = (float)__popcll(__ballot(repeats)) / 64.0f;
    return (wave + 10.0f * runs) * (float)h.pardeg > lanes;
}

template <typename T>
union DecLongLds {
    struct {
        uint32_t cells[dec_waves<T>()][DEC_CELLS + 4];
        uint4 out[dec_waves<T>()][DEC_SUBLEN_MAX * sizeof(T) / 16];
    } wave;
    struct {
        uint4 ring[DECL_WAVES][64 * 4];
        uint32_t strip[DECL_WAVES][64 * 8 * sizeof(T)];
    } lane;
};

// Long streams: huf_dec_kernel's waves, or the first DECL_WAVES of them with a
// partition per lane; one launch for both, as only the stream says which (the
// LDS and the 78 registers of either leave room for three workgroups per CU; a
// table build in each branch, as one before both spilled scalars).
template <typename T>
__global__ void __launch_bounds__(64 * dec_waves<T>())
huf_dec_long_kernel(const uint8_t* __restrict__ in, uint64_t in_bytes, T* __restrict__ out, uint64_t n,
                    int* __restrict__ d_status) {
    static_assert(sizeof(T) <= 2, "the tables hold the symbols of 1- and 2-byte keys");
    constexpr uint32_t WAVES = dec_waves<T>();
    __shared__ DecLds s_tab;
    __shared__ DecLongLds<T> s;
    DecHead h;
    if (!dec_head<T>(in, in_bytes, n, h)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *d_status = 1;
        return;
    }
    const T* keys = reinterpret_cast<const T*>(in + h.e1 + 256);
    const uint32_t w = wave_in_wg();
    if (!dec_by_lanes<T>(h, n)) {
        if (blockIdx.x >= DEC_MAX_BLOCKS) return;
        const DecTables tb = dec_build<T, 64 * WAVES>(in, h, s_tab);
        const uint32_t stride = min(gridDim.x, DEC_MAX_BLOCKS) * WAVES;
        for (uint32_t p = blockIdx.x * WAVES + w; p < h.pardeg; p += stride)
            dec_wave<T>(h, tb, keys, p, n, out, s.wave.cells[w], s.wave.out[w], d_status);
        return;
    }
    if (blockIdx.x * DECL_WAVES * 64 >= h.pardeg) return;
    const DecTables tb = dec_build<T, 64 * WAVES>(in, h, s_tab);
    if (w >= DECL_WAVES) return;
    for (uint32_t p0 = (blockIdx.x * DECL_WAVES + w) * 64; p0 < h.pardeg; p0 += gridDim.x * DECL_WAVES * 64) {
        const uint32_t p = p0 + (uint32_t)lane_id();
        const bool bad = p < h.pardeg && (uint64_t)h.par_entry[p] + ((uint64_t)h.par_nbit[p] + 31) / 32 > h.ncells;
        if (__ballot(bad)) {  // cells past the end: the stream is refused
            if (lane_id() == 0) *d_status = 1;
            continue;
        }
        dec_lanes<T>(h, tb, keys, p0, n, out, reinterpret_cast<uint32_t*>(s.lane.ring[w]), s.lane.strip[w], d_status);
    }
}

struct EncWs {
    size_t pardeg, o_ncell, o_tot, o_nbit, o_scan, o_cells, total;
};
EncWs enc_layout(size_t n, int sl) {
    EncWs w;
    w.pardeg = cdiv(std::max<size_t>(n, 1), (size_t)sl);
    size_t o = 0;
    w.o_ncell = o; o = align_up(o + 4 * w.pardeg, 256);
    w.o_tot = o;   o = align_up(o + 256, 256);  // total cells (u32)
    w.o_nbit = o;  o = align_up(o + 8 * NBIT_SLOTS, 256);  // bit-total accumulators (u64)
    w.o_scan = o;  o = align_up(o + scan_ws_bytes(w.pardeg), 256);
    w.o_cells = o; o = align_up(o + 4 * (size_t)cells_of(sl) * w.pardeg, 256);
    w.total = o;
    return w;
}

template <typename T, int SL>
int enc_impl(hipStream_t s, const void* in, size_t n, uint32_t bklen, const uint32_t* bk4, const uint8_t* rev,
             void* out, size_t cap, void* copy, uint64_t* out_size, void* ws, size_t ws_bytes) {
    constexpr int CELLS = cells_of(SL);
    const EncWs L = enc_layout(n, SL);
    if (ws_bytes < L.total) return fail(FZH_E_CAPACITY, "huffman enc: workspace too small");
    if (n == 0) return fail(FZH_E_INVALID, "huffman enc: empty input");
    if (n > 0x7FFFFFFFull * SL) return fail(FZH_E_INVALID, "huffman enc: input too large");
    if (cap < fzh_huffman_enc_bound(n, bklen, sizeof(T))) return fail(FZH_E_CAPACITY, "huffman enc: output below bound");
    const uint32_t rev_bytes = (uint32_t)fzh_huffman_revbook_bytes(bklen, sizeof(T));
    if (rev_bytes % 4) return fail(FZH_E_INVALID, "huffman enc: bklen * sizeof(T) must be a multiple of 4");
    if (((uintptr_t)out | (uintptr_t)copy) % 16) return fail(FZH_E_INVALID, "huffman enc: output must be 16-byte aligned");
    const uint32_t pardeg = (uint32_t)L.pardeg;
    const uint32_t ent1 = HDR_BYTES, ent2 = ent1 + rev_bytes, ent3 = ent2 + 4 * pardeg, ent4 = ent3 + 4 * pardeg;
    uint8_t* w = (uint8_t*)ws;
    uint32_t* ncell = (uint32_t*)(w + L.o_ncell);
    uint32_t* tot = (uint32_t*)(w + L.o_tot);
    uint32_t* scells = (uint32_t*)(w + L.o_cells);
    uint8_t* o8 = (uint8_t*)out;
    const bool book_in_lds = bklen <= 8192;
    const size_t lds = (size_t)4 * CELLS * 4 + (book_in_lds ? 4 * (size_t)bklen : 0);
    const unsigned blocks = (unsigned)cdiv(pardeg, 4);
    const unsigned eb = book_in_lds ? std::min(blocks, ENC_BLOCKS) : blocks;
    if (book_in_lds)
        launch_k("huf_enc_kernel", huf_enc_kernel<T, SL, true>, dim3(eb), dim3(256), (uint32_t)lds, s, (const T*)in, n,
                 bklen, bk4, rev, rev_bytes, o8, scells, ncell, pardeg);
    else
        launch_k("huf_enc_kernel", huf_enc_kernel<T, SL, false>, dim3(eb), dim3(256), (uint32_t)lds, s, (const T*)in,
                 n, bklen, bk4, rev, rev_bytes, o8, scells, ncell, pardeg);
    if (int rc = scan_u32(s, ncell, reinterpret_cast<uint32_t*>(o8 + ent3), pardeg, nullptr, tot, w + L.o_scan))
        return rc;
    unsigned long long* nbit_acc = reinterpret_cast<unsigned long long*>(w + L.o_nbit);
    launch_k("huf_pack_kernel", huf_pack_kernel, dim3(blocks), dim3(256), 0, s, scells, ncell, o8, (uint8_t*)copy, ent1,
             ent2, ent3, ent4, pardeg, (uint32_t)CELLS, nbit_acc);
    launch_k("huf_header_kernel", huf_header_kernel, dim3(1), dim3(256), 0, s, o8, (uint8_t*)copy, n, bklen, (uint32_t)SL,
             ent1, ent2, ent3, ent4, pardeg, tot, out_size, nbit_acc);
    FZH_CHECK_LAUNCH("huffman encode");
    return FZH_OK;
}

template <int SL>
int encode_sl(hipStream_t s, const void* d_in, size_t n, int elem_bytes, uint32_t bklen, const uint32_t* d_bk4,
              const uint8_t* d_revbook, void* d_out, size_t out_cap, void* d_copy, uint64_t* d_out_size, void* d_ws,
              size_t ws_bytes) {
    if (ws_bytes < std::max(enc_layout(n, SUBLEN).total, enc_layout(n, SUBLEN_FINE).total)) return fail(FZH_E_CAPACITY, "huffman enc: workspace too small");
    switch (elem_bytes) {
    case 1: return enc_impl<uint8_t, SL>(s, d_in, n, bklen, d_bk4, d_revbook, d_out, out_cap, d_copy, d_out_size, d_ws, ws_bytes);
    case 2: return enc_impl<uint16_t, SL>(s, d_in, n, bklen, d_bk4, d_revbook, d_out, out_cap, d_copy, d_out_size, d_ws, ws_bytes);
    case 4: return enc_impl<uint32_t, SL>(s, d_in, n, bklen, d_bk4, d_revbook, d_out, out_cap, d_copy, d_out_size, d_ws, ws_bytes);
    default: return fail(FZH_E_INVALID, "huffman enc: elem_bytes must be 1, 2 or 4");
    }
}

}  // namespace

int huffman_encode(hipStream_t s, bool fine, const void* d_in, size_t n, int elem_bytes, uint32_t bklen,
                   const uint32_t* d_bk4, const uint8_t* d_revbook, void* d_out, size_t out_cap, void* d_copy,
                   uint64_t* d_out_size, void* d_ws, size_t ws_bytes) {
    return (fine ? encode_sl<SUBLEN_FINE> : encode_sl<SUBLEN>)(s, d_in, n, elem_bytes, bklen, d_bk4, d_revbook, d_out,
                                                               out_cap, d_copy, d_out_size, d_ws, ws_bytes);
}
}  // namespace fzh

using namespace fzh;

extern "C" {

int fzh_histogram(void* stream, const void* d_in, size_t n, int elem_bytes, uint32_t bklen, uint32_t* d_freq) {
    if (bklen == 0) return fail(FZH_E_INVALID, "histogram: bklen must be > 0");
    if (int rc = zero_bytes(S(stream), d_freq, 4 * (size_t)bklen)) return rc;
    if (n == 0) return FZH_OK;
    if ((uintptr_t)d_in % 16) return fail(FZH_E_INVALID, "histogram: input must be 16-byte aligned");
    const int replicas = bklen <= 1024 ? 8 : (bklen <= 4096 ? 4 : (bklen <= 16384 ? 1 : 0));
    const uint32_t rs = replicas == 8 ? bklen + 1 : bklen;  // replica stride in words (LDS <= 64 KiB)
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(cdiv(n, 256 * 64), 1024));
    hipStream_t s = S(stream);
#define FZH_HIST(T)                                                                                       \
    if (replicas)                                                                                         \
        launch_k("hist_kernel", hist_kernel<T>, dim3(blocks), dim3(256), (uint32_t)(4 * rs * replicas), s, (const T*)d_in, n, bklen, d_freq, replicas); \
    else                                                                                                  \
        launch_k("hist_global_kernel", hist_global_kernel<T>, dim3(blocks), dim3(256), 0, s, (const T*)d_in, n, bklen, d_freq);
    switch (elem_bytes) {
    case 1: FZH_HIST(uint8_t) break;
    case 2: FZH_HIST(uint16_t) break;
    case 4: FZH_HIST(uint32_t) break;
    default: return fail(FZH_E_INVALID, "histogram: elem_bytes must be 1, 2 or 4");
    }
#undef FZH_HIST
    FZH_CHECK_LAUNCH("hist_kernel");
    return FZH_OK;
}

size_t fzh_huffman_enc_bound(size_t n, uint32_t bklen, int elem_bytes) {
    const size_t pardeg = cdiv(std::max<size_t>(n, 1), SUBLEN);
    // every codeword is at most 28 bits
    return HDR_BYTES + fzh_huffman_revbook_bytes(bklen, elem_bytes) + 8 * pardeg + 4 * cdiv(n * 28, 32) + 4 * pardeg + 64;
}

size_t fzh_huffman_enc_ws_bytes(size_t n) {
    return std::max(enc_layout(n, SUBLEN).total, enc_layout(n, SUBLEN_FINE).total);
}

int fzh_huffman_encode(void* stream, const void* d_in, size_t n, int elem_bytes, uint32_t bklen,
                       const uint32_t* d_bk4, const uint8_t* d_revbook, void* d_out, size_t out_cap,
                       uint64_t* d_out_size, void* d_ws, size_t ws_bytes) {
    return huffman_encode(S(stream), false, d_in, n, elem_bytes, bklen, d_bk4, d_revbook, d_out, out_cap, nullptr,
                          d_out_size, d_ws, ws_bytes);
}

int fzh_huffman_encode_fine(void* stream, const void* d_in, size_t n, int elem_bytes, uint32_t bklen,
                            const uint32_t* d_bk4, const uint8_t* d_revbook, void* d_out, size_t out_cap,
                            uint64_t* d_out_size, void* d_ws, size_t ws_bytes) {
    return huffman_encode(S(stream), true, d_in, n, elem_bytes, bklen, d_bk4, d_revbook, d_out, out_cap, nullptr,
                          d_out_size, d_ws, ws_bytes);
}

int fzh_huffman_decode(void* stream, const void* d_in, size_t in_bytes, int elem_bytes, void* d_out, size_t n,
                       int* d_status) {
    if (n == 0) return FZH_OK;
    if (!d_status) return fail(FZH_E_INVALID, "huffman dec: null status");
    if ((uintptr_t)d_in % 4 || (uintptr_t)d_out % 16) return fail(FZH_E_INVALID, "huffman dec: input 4-byte, output 16-byte alignment required");
    // the partition count is in the stream; the coarse 768-symbol partitions
    // bound it
    const size_t pardeg = cdiv(n, SUBLEN);
    hipStream_t s = S(stream);
#define FZH_HUF_DEC(T)                                                                                         \
    if (sizeof(T) <= 2 && pardeg >= DECL_MIN_PARTS) {                                                          \
        using U = std::conditional_t<sizeof(T) <= 2, T, uint16_t>;                                             \
        const unsigned blocks = (unsigned)std::min<size_t>(                                                    \
            std::max<size_t>(cdiv(pardeg, 64 * DECL_WAVES), DEC_MAX_BLOCKS), 65536);                           \
        launch_k("huf_dec_long_kernel", huf_dec_long_kernel<U>, dim3(blocks), dim3(64 * dec_waves<U>()), 0, s, \
                 (const uint8_t*)d_in, in_bytes, (U*)d_out, n, d_status);                                      \
    } else {                                                                                                   \
        const unsigned blocks = (unsigned)std::min<size_t>(cdiv(pardeg, dec_waves<T>()), DEC_MAX_BLOCKS);     \
        launch_k("huf_dec_kernel", huf_dec_kernel<T>, dim3(blocks), dim3(64 * dec_waves<T>()), 0, s,          \
                 (const uint8_t*)d_in, in_bytes, (T*)d_out, n, d_status);                                      \
    }
    switch (elem_bytes) {
    case 1: FZH_HUF_DEC(uint8_t) break;
    case 2: FZH_HUF_DEC(uint16_t) break;
    case 4: FZH_HUF_DEC(uint32_t) break;
    default: return fail(FZH_E_INVALID, "huffman dec: elem_bytes must be 1, 2 or 4");
    }
#undef FZH_HUF_DEC
    FZH_CHECK_LAUNCH("huf_dec_kernel");
    return FZH_OK;
}

}  // extern "C"
