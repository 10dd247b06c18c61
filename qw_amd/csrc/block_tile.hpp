// block_tile.hpp - the key tile that the block kernels keep in LDS: its shape
// and layouts, shared by the cache kernel (attend_block.hip) and the row
// kernel (attend_rows.hip), which reads the same tile images.
#pragma once

#include "qw_common.hpp"

namespace qw {

template <int D>
struct BlockShape {
    static constexpr int KT = 16384 / D;  // keys a tile (64 at D=256, 128 at D=128)
    static constexpr int NSUB = KT / 32;  // 32-key sub-blocks a tile
    static constexpr int NM = D / 32;     // QK MFMAs per 16-key tile
    static constexpr int NT = D / 16;     // P.V MFMAs (16-dim output tiles)
    static constexpr int NG = D / 64;     // affine groups a row
    static constexpr int TPR = D / 32;    // 32-dim K slices a row
    static constexpr int LTPR = TPR == 8 ? 3 : TPR == 4 ? 2 : 1;
    static constexpr int TPB = D / 4;     // 4-slot V slices a block
    static constexpr int KBUF = (D / 8) * KT * 16;  // K tile bytes in LDS (chunk-major)
    static constexpr int VROW = D + D / 16;  // V block stride in chunks (a pad chunk per 16 slots)
    static constexpr int VBUF = (KT / 8) * VROW * 16;               // V tile bytes in LDS
    static constexpr int BUF = KBUF + VBUF;                         // one buffer
};

// LDS layouts (16-byte chunks). Measured on gfx950 (ds_read_b128, 8 waves a
// CU): an instruction runs at full rate (~210 B/clk a CU) when the 16 lanes of
// each quarter-wave hit 16 distinct bank groups (chunk mod 16) AND lane r of
// every quarter-wave hits the same bank group; quarter-waves whose bank groups
// are rotated against each other run at ~125 B/clk, like a 2-way conflict.
//   K  chunk-major [D/8 chunks][KT keys]: chunk c of key k sits at
//      kaddr(k, c) = c * KT + swz(k), swz(k) = k ^ (bit 4 of k) << 2. The QK
//      A operand (lane (g, r), r = lane & 15) reads chunk g + 4m of key
//      8(r>>2) + 4t + (r&3) + 32u: the chunk stride KT keeps the quarter-waves
//      g aligned, and swz maps the 16 keys of a quarter-wave (k mod 16 takes
//      0-3 and 8-11 twice) to 16 distinct bank groups. Every (step, sub-block)
//      is the lane's base (one a 16-key tile t) plus an immediate. The store
//      phase gives each quarter-wave 16 consecutive keys of one 32-dim slice
//      (quarter-waves differ in the slice): also aligned and distinct.
//   V  [8-key block][D slots + D/16 pad][8 keys], slots in the V plane's
//      physical dim order, slot s at s + (s >> 4): the P.V B operand reads 16
//      consecutive slots a phase (slot 16mm + r at 17mm + r, an immediate
//      per mm), and the store phase's lanes (slots 4j + e) land on 16 distinct
//      bank groups.
__device__ __forceinline__ int kswz(int key) { return key ^ (((key >> 4) & 1) << 2); }
template <int KT>
__device__ __forceinline__ int kaddr(int key, int chunk) {
    return chunk * KT + kswz(key);
}


// max / sum of v over the lane pair (l, l ^ 16), then over (l, l ^ 32): row
// swaps in the VALU (v_permlane16/32_swap) instead of LDS permutes.
__device__ __forceinline__ float wave_max_g(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float wave_sum_g(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Bits that keep the first n keys of an 8-key piece of V (key e in half e) and zero the
// others: a hidden key has weight 0 in P . V, but 0 x inf is NaN.
__device__ __forceinline__ u32x4 keep_keys(int n) {
    u32x4 m;
#pragma unroll
    for (int j = 0; j < 4; j++) m[j] = (2 * j < n ? 0xFFFFu : 0u) | (2 * j + 1 < n ? 0xFFFF0000u : 0u);
    return m;
}

// An explicit mask in a key tile: a lane's 8 consecutive keys of one row, from
// element offset off of a mask with key stride 1 (any alignment), n of them inside
// the mask (n <= 0: none); raw, so that the loads can be issued ahead of the MFMAs.
__device__ __forceinline__ void mask_load8(const void* mask, int dtype, int64_t off, int n,
                                           u32x4 (&raw)[2]) {
    raw[0] = raw[1] = u32x4{0, 0, 0, 0};
    if (dtype == QW_MASK_BOOL) {
        const uint8_t* p = (const uint8_t*)mask + off;
        if (n >= 8) {
            u32x2 w;
            __builtin_memcpy(&w, p, 8);
            raw[0].x = w.x;
            raw[0].y = w.y;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (e < n) raw[0][e >> 2] |= (uint32_t)p[e] << (8 * (e & 3));
        }
    } else if (dtype == QW_DTYPE_F32) {
        const uint32_t* p = (const uint32_t*)mask + off;
        if (n >= 8) {
            __builtin_memcpy(&raw[0], p, 16);
            __builtin_memcpy(&raw[1], p + 4, 16);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (e < n) raw[e >> 2][e & 3] = p[e];
        }
    } else {
        const uint16_t* p = (const uint16_t*)mask + off;
        if (n >= 8) {
            __builtin_memcpy(&raw[0], p, 16);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (e < n) raw[0][e >> 1] |= (uint32_t)p[e] << (16 * (e & 1));
        }
    }
}
// Key e of them: whether a bool mask hides it; an additive mask's term, cast to
// fp16 as the reference casts float masks.
__device__ __forceinline__ bool mask_hides(const u32x4 (&raw)[2], int e) {
    return ((raw[0][e >> 2] >> (8 * (e & 3))) & 0xFFu) == 0;
}
__device__ __forceinline__ f16 mask_term(const u32x4 (&raw)[2], int dtype, int e) {
    const uint32_t w = raw[0][e >> 1] >> (16 * (e & 1));
    if (dtype == QW_DTYPE_F32) return (f16)__uint_as_float(raw[e >> 2][e & 3]);
    if (dtype == QW_DTYPE_BF16) return (f16)__uint_as_float(w << 16);
    return __builtin_bit_cast(f16, (uint16_t)w);
}

}  // namespace qw
