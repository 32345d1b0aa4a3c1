// fzh_huffman_enc.h — one partition's Huffman codewords packed by one wave,
// shared by the single-stream encoder (huffman.hip) and the batched one
// (batch.hip).
#pragma once

#include "fzh_internal.h"

namespace fzh {
namespace {

constexpr int SUBLEN = 768;       // coarse partitions
constexpr int SUBLEN_FINE = 1024; // fine partitions
constexpr int HDR_BYTES = 128;

// cells per partition slot (every codeword is at most 28 bits)
constexpr int cells_of(int sl) { return (sl * 28 + 31) / 32 + 2; }

// Packs the cnt (<= SL) symbols at `src` MSB-first into `cells` (LDS,
// cells_of(SL) words of this wave) and returns their bit count.  A lane takes
// SL / 64 consecutive symbols: their lengths add up in the lane, so one wave
// scan places all of them, and their codes are shifted together in a register
// that goes to LDS a whole cell at a time (about two OR operations per lane
// and 12 symbols of 6.5 bits).  With symbols strided by 64 over the lanes
// every symbol took a wave scan and one or two LDS ORs that collide with its
// neighbours' in the same cell: 2^27 symbols 234 us, now 96.
// wide: src is aligned to the lane's vector loads; the codebook is s_bk in
// LDS (BOOK_LDS) or bk4 in memory.  (A template parameter, not a pointer
// chosen at run time: a pointer that may be either makes every lookup a FLAT
// access.)
template <typename T, int SL>
constexpr int enc_load_bytes() {
    constexpr int B = SL / 64 * (int)sizeof(T);
    return B % 16 == 0 ? 16 : (B % 8 == 0 ? 8 : 4);
}

template <typename T, int SL, bool BOOK_LDS>
__device__ __forceinline__ uint32_t huf_encode_partition(const T* __restrict__ src, uint32_t cnt, bool wide,
                                                         const uint32_t* s_bk, const uint32_t* __restrict__ bk4,
                                                         uint32_t bklen, uint32_t* cells) {
    constexpr int K = SL / 64;  // symbols per lane
    constexpr int B = K * (int)sizeof(T);
    constexpr int V = enc_load_bytes<T, SL>();
    const int l = lane_id();
    // lane l: symbols K l .. K l + K - 1 of the partition
    T sym[K];
    if (cnt == SL && wide) {
        const T* a = src + K * l;
#pragma unroll
        for (int i = 0; i < B / V; i++) {
            if constexpr (V == 16)
                reinterpret_cast<uint4*>(sym)[i] = gld_u4(reinterpret_cast<const uint4*>(a) + i);
            else if constexpr (V == 8) {
                const fzh_u32x2 w = *gp(reinterpret_cast<const fzh_u32x2*>(a) + i);
                reinterpret_cast<uint2*>(sym)[i] = make_uint2(w.x, w.y);
            } else
                reinterpret_cast<uint32_t*>(sym)[i] = *gp(reinterpret_cast<const uint32_t*>(a) + i);
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; k++) sym[k] = K * l + k < (int)cnt ? *gp(src + K * l + k) : (T)0;
    }
    uint32_t word[K], bits = 0;  // length << 27 | code
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint32_t x = (uint32_t)sym[k];
        // a symbol past the partition's end or out of range (reported by the caller) gets no code
        const bool ok = x < bklen && (cnt == SL || K * l + k < (int)cnt);
        word[k] = ok ? (BOOK_LDS ? s_bk[x] : bk4[x]) : 0u;
        bits += word[k] >> 27;
    }
    const uint32_t incl = wave_incl_scan(bits);
    const uint32_t nbit = lane63(incl);
    const uint32_t ncell = (nbit + 31) / 32;
    for (uint32_t i = l; i <= ncell; i += 64) cells[i] = 0u;
    wave_lds_sync();
    // the lane's codes shifted into place; a cell leaves the register when it
    // is full, and what lanes share of a cell is ORed together in LDS
    uint32_t at = (incl - bits) >> 5, fill = (incl - bits) & 31u, hi = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint32_t c = word[k] & 0x07FFFFFFu;
        const uint32_t to = fill + (word[k] >> 27);  // 0 .. 62
        const uint32_t x = __builtin_amdgcn_alignbit(c, 0u, to);  // c << (32 - to % 32), 0 if that is 32
        if (to >= 32) {
            atomicOr(&cells[at], hi | (c >> (to & 31u)));
            at++;
        }
        hi = to >= 32 ? x : hi | x;
        fill = to & 31u;
    }
    if (fill) atomicOr(&cells[at], hi);
    wave_lds_sync();
    return nbit;
}

}  // namespace
}  // namespace fzh
