// attend_rows.hip - attention of many query rows over key tiles that are laid
// out once: fp16 K/V views of the caller, gfx950.
//
// Reference path replaced: layers::attention (crates/mlxcel-core/src/layers.rs:
// 4010-4060) and causal_attention (crates/mlxcel-core/src/lib.rs:3185-3275) over
// fp16 K/V that the caller holds, with a sliding window, a softcap or an
// explicit mask. Semantics are those of sdpa_general.hip, which keeps the calls
// of few rows (the dispatch there says where the line lies and why):
//   softcap == 0: S = f16(f16(f16(scale) q) . k), an additive mask cast to fp16
//     and added in fp16, softmax in fp32, P in fp16;
//   softcap > 0: S = f16(q . k), s = tanh(S scale / cap) cap in fp32, the mask
//     added in fp32, softmax in fp32, P.V with fp32 P (an fp16 high part and an
//     fp16 remainder, two MFMAs).
//
// Two launches (three when the keys are split):
//   rows_image_kernel writes each key tile (16384 / D keys) of each KV head in
//     the LDS layout of block_tile.hpp, once;
//   rows_attend_kernel: a workgroup owns NW waves x 16 rows (row index r * G +
//     head in group) and runs over the tiles, copying each tile's image into one
//     of two LDS buffers by LDS-DMA while it computes the other. A wave forms
//     S^T = K . Q^T with v_mfma_f32_16x16x32_f16 (A = K rows), which leaves each
//     lane 8 consecutive keys of one row, the A operand of P . V;
//   the split-K merge of attend_decode.hip. The partials are fp32.
// What bounds it: the LDS operand reads (one 1 KB read an MFMA) and the MFMAs;
// laying the tiles out costs one read and one write of K and V. Before, every
// workgroup of 64 rows transposed V into LDS with 2-byte stores and rescaled
// its accumulators every 32 keys. Measured: see sdpa_takes_rows in sdpa_general.hip.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "block_tile.hpp"
#include "kv_cache.hpp"
#include "qw_common.hpp"

namespace qw {

namespace {

struct RowsArgs {
    const f16* q;    // [hq][Tq][D]
    f16* out;        // [hq][Tq][D], written directly by unsplit workgroups
    float* part_o;   // [hkv][n_split][PR][D] in V slot order, rows from prow0
    float2* part_ml; // [hkv][n_split][PR]
    const char* img; // [hkv][n_tiles - tile0][BUF]: the images of tiles tile0 ..
    int T, Tq, G, R, hkv, n_tiles, tile0, causal;
    int window;      // > 0: keys p - window + 1 .. p of the row at position p
    // The first n_main workgroups are unsplit query tiles (unit u: tile u / hkv,
    // head u % hkv); the others are splits of the query tiles from qt0 on (unit
    // t: split t % n_split, head (t / n_split) % hkv, tile qt0 + t / (n_split hkv)),
    // tiles_per_split key tiles each. The dispatcher starts the split ones as the
    // first ones end.
    int n_main, qt0, n_split, tiles_per_split, prow0, PR;
    const void* mask;  // [hq or broadcast][Tq][T], key stride 1
    int mask_dtype;    // QW_MASK_BOOL / QW_DTYPE_*
    int64_t mhs, mrs;
    float scale_h;
    Softcap softcap;
};

// fp16 K/V rows with strides -> images of the tiles from tile0 on. grid (tiles,
// KV heads). A thread
// takes the 32-dim slice of one key of K (quarter-waves of 16 keys, as
// block_tile.hpp's store rule asks) and 4 dims of an 8-key block of V (64 lanes
// read whole rows; the 8 x 4 piece is transposed in registers).
template <int D>
__global__ __launch_bounds__(512) void rows_image_kernel(const f16* __restrict__ k,
                                                         const f16* __restrict__ v, int64_t khs,
                                                         int64_t krs, int64_t vhs, int64_t vrs,
                                                         int T, int tile0, char* __restrict__ img) {
    using S = BlockShape<D>;
    constexpr int KT = S::KT;
    extern __shared__ __attribute__((aligned(16))) char lds_buf[];
    half8* const sK = (half8*)lds_buf;
    half8* const sV = (half8*)(lds_buf + S::KBUF);
    const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, t0 = (tile0 + t) * KT;
    static_assert(KT * S::TPR == 512 && (KT / 8) * S::TPB == 512, "one slice of each kind a thread");
    const int q32 = (tid >> 4) & (S::TPR - 1), kk = (tid & 15) | ((tid >> (4 + S::LTPR)) << 4);
    const int vb = tid / S::TPB, vj = tid % S::TPB;
    u32x4 kc[4] = {};
    if (t0 + kk < T) {
        const u32x4* src = (const u32x4*)(k + h * khs + (int64_t)(t0 + kk) * krs + 32 * q32);
#pragma unroll
        for (int w = 0; w < 4; w++) kc[w] = src[w];
    }
    half4v vr[8] = {};
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (t0 + 8 * vb + i < T)
            vr[i] = *(const half4v*)(v + h * vhs + (int64_t)(t0 + 8 * vb + i) * vrs + 4 * vj);
#pragma unroll
    for (int w = 0; w < 4; w++) sK[kaddr<KT>(kk, 4 * q32) + w * KT] = as_h8(kc[w]);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        half8 y;
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = vr[i][e];
        const int sl = v_phys_dim(4 * vj + e, D, 16);
        sV[vb * S::VROW + sl + (sl >> 4)] = y;
    }
    __syncthreads();
    char* dst = img + ((int64_t)h * gridDim.x + t) * S::BUF;
    for (int i = 16 * tid; i < S::BUF; i += 16 * 512) *(u32x4*)(dst + i) = *(const u32x4*)(lds_buf + i);
}

// NW: 12 waves (three a SIMD) for calls of many rows without a mask, else 8.
template <int D, int NW, bool CAP, bool MASK>
__global__ __launch_bounds__(64 * NW, 1) void rows_attend_kernel(RowsArgs a) {
    using S = BlockShape<D>;
    constexpr int KT = S::KT, NSUB = S::NSUB, NM = S::NM, NT = S::NT, BUF = S::BUF, KBUF = S::KBUF;
    constexpr int VROW = S::VROW;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    int sp = 0, qt, h, n_split = 1, tps = a.n_tiles;
    {
        const int lin = blockIdx.x;
        if (lin < a.n_main) {
            qt = lin / a.hkv;
            h = lin % a.hkv;
        } else {
            const int t = lin - a.n_main;
            n_split = a.n_split;
            tps = a.tiles_per_split;
            sp = t % n_split;
            h = (t / n_split) % a.hkv;
            qt = a.qt0 + t / (n_split * a.hkv);
        }
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int row0 = qt * 16 * NW, row_last = min(a.R, row0 + 16 * NW) - 1;
    const int wrow0 = row0 + 16 * wave;
    const int pos0 = a.T - a.Tq;  // position of query row 0
    // the workgroup's tiles: its split of those that some row of it sees
    const int wg_lim = a.causal ? pos0 + row_last / a.G : a.T - 1;
    const int t_win = a.window > 0 ? max(0, pos0 + row0 / a.G - a.window + 1) / KT : 0;
    const int t0 = t_win + sp * tps, t1 = min(min(a.n_tiles, t0 + tps), wg_lim / KT + 1);
    // key limits: of the wave's last row (tiles past it are skipped), of its
    // first (tiles past it need the compares); window starts likewise
    const bool wave_live = wrow0 < a.R;
    const int wave_last = min(a.R, wrow0 + 16) - 1;
    const int wave_lim = a.causal ? pos0 + wave_last / a.G : a.T - 1;
    const int wave_first_lim = a.causal ? pos0 + wrow0 / a.G : a.T - 1;
    const int wave_lo_max = a.window > 0 ? pos0 + wave_last / a.G - a.window + 1 : 0;
    const int wave_lo_min = a.window > 0 ? pos0 + wrow0 / a.G - a.window + 1 : 0;
    const int rho = wrow0 + r16;
    const bool row_ok = rho < a.R;
    const int r = row_ok ? rho / a.G : 0, qh = h * a.G + (row_ok ? rho - r * a.G : 0);
    const int lim = !row_ok ? -1 : a.causal ? pos0 + r : a.T - 1;
    const int wlo = a.window > 0 ? pos0 + r - a.window + 1 : 0;
    half8 qb[NM];
    {
        const f16* qrow = a.q + ((int64_t)qh * a.Tq + r) * D;
        const f16 sc = row_ok ? (CAP ? (f16)1.0f : (f16)a.scale_h) : (f16)0.0f;
#pragma unroll
        for (int m = 0; m < NM; m++) {
            half8 x = *(const half8*)(qrow + 32 * m + 8 * g);
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = x[e] * sc;
            qb[m] = x;
        }
    }
    const int64_t moff = MASK ? (int64_t)qh * a.mhs + (int64_t)r * a.mrs : 0;

    float m_run = -INFINITY, l_run = 0.0f;  // softmax reference, this lane's share of the sum
    float4v acc_o[NT];
#pragma unroll
    for (int mm = 0; mm < NT; mm++) acc_o[mm] = float4v{0.f, 0.f, 0.f, 0.f};

    // NU sub-blocks of 32 keys (all of a tile's, but half of D = 64's eight, whose
    // scores would not fit the registers) from sub-block ub of buffer b, whose
    // first key is kt0
    constexpr int NU = NSUB < 4 ? NSUB : 4;
    // EDGE: keys that some row of the workgroup does not see are among the tile's
    auto tile = [&](int b, int ub, int kt0, auto edge_c) {
        constexpr bool EDGE = decltype(edge_c)::value;
        const half8* sK8 = (const half8*)(lds + BUF * b) + 32 * ub;
        const half8* sV8 = (const half8*)(lds + BUF * b + KBUF) + 4 * ub * VROW;
        // the lane's 8 mask entries of each 32-key sub-block, raw (key stride 1,
        // any alignment), requested before the MFMAs that hide them
        u32x4 raw[MASK ? NU : 1][2];
        if constexpr (MASK) {
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const int t = kt0 + 32 * u + 8 * g;
                const int n = row_ok ? min(8, a.T - t) : 0;
                mask_load8(a.mask, a.mask_dtype, moff + t, n, raw[u]);
            }
        }
        // S^T: A row r16 of 16-key MFMA tile (u, tt) is key 32u + 8(r16>>2) + 4tt +
        // (r16&3), so lane (g, r16) gets keys 32u + 8g + e (e = 4tt + i) of row r16
        const int key0 = 8 * (r16 >> 2) + (r16 & 3);
        const int b4 = (key0 >> 4) & 1;
        const half8* kbase0 = sK8 + g * KT + key0 + 4 * b4;
        const half8* kbase1 = sK8 + g * KT + key0 + 4 * (b4 ^ 1);
        float4v acc[NU][2];
#pragma unroll
        for (int u = 0; u < NU; u++) acc[u][0] = acc[u][1] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const half8 ka = kbase0[4 * m * KT + 32 * u], kb2 = kbase1[4 * m * KT + 32 * u];
                acc[u][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qb[m], acc[u][0], 0, 0, 0);
                acc[u][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kb2, qb[m], acc[u][1], 0, 0, 0);
            }
        // four LDS reads kept ahead of the MFMAs (as in attend_block.hip)
        {
            constexpr int NQ = NM * NU * 2, AH = 4;
            __builtin_amdgcn_sched_group_barrier(0x100, AH, 0);
#pragma unroll
            for (int i = 0; i < NQ - AH; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, AH, 0);
        }
        const bool edge = EDGE && (kt0 + 32 * NU - 1 > wave_first_lim || (a.window > 0 && kt0 < wave_lo_max));
        half8 pop[NU], popl[CAP ? NU : 1];
        // fp16 scores (softcap: fp32), masked
        half2v sh[CAP ? 1 : NU][4];
        float sf[CAP ? NU : 1][8];
        if constexpr (CAP) {
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int e = 0; e < 8; e++) sf[u][e] = (float)(f16)acc[u][e >> 2][e & 3];
            a.softcap.apply(sf);
        } else {
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int e = 0; e < 8; e++) sh[u][e >> 1][e & 1] = (f16)acc[u][e >> 2][e & 3];
        }
        auto hide = [&](int u, int e) {
            if constexpr (CAP) sf[u][e] = -INFINITY;
            else sh[u][e >> 1][e & 1] = (f16)(-INFINITY);
        };
        if constexpr (MASK) {
            if (a.mask_dtype == QW_MASK_BOOL) {
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (mask_hides(raw[u], e)) hide(u, e);
            } else {
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const f16 ad = mask_term(raw[u], a.mask_dtype, e);
                        if constexpr (CAP)
                            sf[u][e] += (float)ad;
                        else
                            sh[u][e >> 1][e & 1] = (f16)((float)sh[u][e >> 1][e & 1] + (float)ad);
                    }
            }
        }
        if (edge) {
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int key = kt0 + 32 * u + 8 * g + e;
                    if (key > lim || key < wlo) hide(u, e);
                }
        }
        // Online softmax. fp16 P goes against the running maximum, as sdpa_general.hip's
        // does, so that the largest weight is exactly 1; the reduction over the row runs
        // only where a lane has a new maximum. (A lazy reference, which moves only past
        // 5.5, rounds that weight too: error against 64 bits 9.50e-4 against 9.45e-4
        // here and in sdpa_general.hip, for 4 % of the time, at 1536 rows over 9.7k keys.)
        // Capped scores enter P . V in two parts, and keep the lazy reference.
        constexpr float kLazy = CAP ? 5.5f : 0.0f;
        float mx;
        if constexpr (CAP) {
            mx = sf[0][0];
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int e = 0; e < 8; e++) mx = fmaxf(mx, sf[u][e]);
        } else {
            half2v m2 = sh[0][0];
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int j = 0; j < 4; j++) m2 = __builtin_elementwise_max(m2, sh[u][j]);
            mx = fmaxf((float)m2.x, (float)m2.y);
        }
        if (__any(mx > m_run + kLazy)) {
            const float m_new = fmaxf(m_run, wave_max_g(mx));
            if (__any(m_run != -INFINITY)) {
                const float alpha =
                    m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m_run - m_new) * kLog2e);
                l_run *= alpha;
                float f[4];
#pragma unroll
                for (int i = 0; i < 4; i++) f[i] = __shfl(alpha, 4 * g + i);
#pragma unroll
                for (int mm = 0; mm < NT; mm++)
#pragma unroll
                    for (int i = 0; i < 4; i++) acc_o[mm][i] *= f[i];
            }
            m_run = m_new;
        }
        const float mref2 = (m_run == -INFINITY ? 0.0f : m_run) * kLog2e;
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x = CAP ? sf[CAP ? u : 0][e] : (float)sh[CAP ? 0 : u][e >> 1][e & 1];
                const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(x, kLog2e, -mref2));
                l_run += p;
                const f16 ph = (f16)p;
                pop[u][e] = ph;
                if constexpr (CAP) popl[u][e] = (f16)(p - (float)ph);
            }
        // O += P . V: B = slot 16mm + r16 of V block 4u + g (keys 32u + 8g .. +7). A key that
        // no row of the wave sees must not enter even with weight 0 (0 x inf is NaN).
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const half8* vb8 = sV8 + (4 * u + g) * VROW + r16;
            u32x4 keep = {};
            if constexpr (EDGE) {
                const int key = kt0 + 32 * u + 8 * g;
                keep = keep_keys(wave_lim + 1 - key) & ~keep_keys(wave_lo_min - key);
            }
#pragma unroll
            for (int mm = 0; mm < NT; mm++) {
                half8 vv = vb8[17 * mm];
                if constexpr (EDGE) vv = as_h8(__builtin_bit_cast(u32x4, vv) & keep);
                acc_o[mm] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pop[u], vv, acc_o[mm], 0, 0, 0);
                if constexpr (CAP)
                    acc_o[mm] = __builtin_amdgcn_mfma_f32_16x16x32_f16(popl[u], vv, acc_o[mm], 0, 0, 0);
            }
        }
        {
            constexpr int NQ = NU * NT, AH = 4, MF = CAP ? 2 : 1;
            __builtin_amdgcn_sched_group_barrier(0x100, AH, 1);
#pragma unroll
            for (int i = 0; i < NQ - AH; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, MF, 1);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, MF * AH, 1);
        }
    };

    // tile t's image into buffer b, 1 KB a wave instruction; M0 is saved and
    // restored so that the compiler's view of it holds (attend_block.hip)
    const char* img0 = a.img + ((int64_t)h * (a.n_tiles - a.tile0) - a.tile0) * BUF;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds;
    static_assert(BUF % 1024 == 0, "a tile buffer is whole 1 KB DMA instructions");
    auto dma = [&](int t, int b) {
        const char* src = img0 + (int64_t)t * BUF + 16 * lane;
        for (int c = wave; c < BUF / 1024; c += NW) {
            uint32_t saved;
            asm volatile(
                "s_mov_b32 %0, m0\n\t"
                "s_mov_b32 m0, %2\n\t"
                "s_nop 0\n\t"
                "global_load_lds_dwordx4 %1, off\n\t"
                "s_nop 0\n\t"
                "s_mov_b32 m0, %0"
                : "=&s"(saved)
                : "v"(src + 1024 * c), "s"(__builtin_amdgcn_readfirstlane(lds0 + BUF * b + 1024 * c))
                : "memory");
        }
    };
    if (t0 < t1) dma(t0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // tiles ta .. tb - 1. The tiles that hold no limit of the workgroup's rows have a loop
    // of their own, without the compares and the masks of V (one loop for both 487 us,
    // this 387, at 1536 rows over 9.7k keys; the masks by a branch spilled registers).
    auto tiles = [&](int ta, int tb, auto edge_c) {
        for (int t = ta; t < tb; t++) {
            const int b = (t - t0) & 1;
            if (t + 1 < t1) dma(t + 1, b ^ 1);
#pragma unroll
            for (int ub = 0; ub < NSUB; ub += NU) {
                const int kt0 = t * KT + 32 * ub;
                if (wave_live && kt0 <= wave_lim && kt0 + 32 * NU > wave_lo_min) tile(b, ub, kt0, edge_c);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
    };
    const int wg_first_lim = a.causal ? pos0 + row0 / a.G : a.T - 1;
    const int wg_lo_max = a.window > 0 ? pos0 + row_last / a.G - a.window + 1 : 0;
    const int t_in = min(t1, max(t0, (max(wg_lo_max, 0) + KT - 1) / KT));  // [t_in, t_out): seen by all rows
    const int t_out = min(t1, max(t_in, (wg_first_lim + 1) / KT));
    tiles(t0, t_in, std::true_type{});
    tiles(t_in, t_out, std::false_type{});
    tiles(t_out, t1, std::true_type{});

    const float lsum = wave_sum_g(l_run);
    if (n_split == 1) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float l = __shfl(lsum, 4 * g + i);
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            const int row = wrow0 + 4 * g + i;
            if (row >= a.R) continue;
            f16* orow = a.out + ((int64_t)(h * a.G + row % a.G) * a.Tq + row / a.G) * D;
            // slot 16mm + r16 is dim NT r16 + mm: a lane's NT dims are consecutive
#pragma unroll
            for (int c = 0; c < NT; c += 4) {
                half4v y;
#pragma unroll
                for (int j = 0; j < 4; j++) y[j] = (f16)(acc_o[c + j][i] * inv);
                *(half4v*)(orow + NT * r16 + c) = y;
            }
        }
    } else {
        const int64_t pbase = ((int64_t)h * n_split + sp) * a.PR - a.prow0;
        if (g == 0 && row_ok) a.part_ml[pbase + rho] = float2{m_run, lsum};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = wrow0 + 4 * g + i;
            if (row >= a.R) continue;
            float* prow = a.part_o + (pbase + row) * D;
#pragma unroll
            for (int mm = 0; mm < NT; mm++) prow[16 * mm + r16] = acc_o[mm][i];
        }
    }
}

template <int D, int NW, bool CAP, bool MASK>
int launch_rows_one(const RowsArgs& a, int grid, hipStream_t stream) {
    const size_t shmem = (size_t)2 * BlockShape<D>::BUF;
    if (int rc = ensure_dynamic_lds((const void*)rows_attend_kernel<D, NW, CAP, MASK>, shmem)) return rc;
    hipLaunchKernelGGL((rows_attend_kernel<D, NW, CAP, MASK>), dim3(grid), dim3(64 * NW), shmem, stream, a);
    QW_HIP_CHECK(hipGetLastError());
    return QW_OK;
}

// How n_qt query tiles of 16 nw rows are spread over 256 CUs: whole rounds of
// unsplit workgroups, the rest split over the keys.
struct RowsPlan {
    int nw, n_qt, q_main, n_split, tps;
    double cost;  // rounds x rows of a round
};

RowsPlan plan_rows(int R, int hkv, int nw, int key_tiles) {
    RowsPlan p{nw, (R + 16 * nw - 1) / (16 * nw), 0, 1, key_tiles, 0.0};
    const int units = p.n_qt * hkv;
    if (units >= 256 && 256 % hkv == 0) p.q_main = units / 256 * (256 / hkv);
    const int tail = (p.n_qt - p.q_main) * hkv;
    double rounds = (double)(p.q_main * hkv) / 256;
    if (tail > 0) {
        // at least two tiles a split: a workgroup's prologue and partials cost about one
        const int want = std::max(1, std::min({256 / tail, (key_tiles + 1) / 2, 256}));
        p.tps = (key_tiles + want - 1) / want;
        p.n_split = (key_tiles + p.tps - 1) / p.tps;
        // (the merge and the partials: about 5 % of a round)
        rounds += (double)((tail * p.n_split + 255) / 256) / p.n_split + (p.n_split > 1 ? 0.05 : 0.0);
    }
    // eight waves a workgroup cost 10 % more a row than twelve (the tile copies
    // and barriers are shared by fewer rows)
    p.cost = rounds * 16 * nw * (nw == 8 ? 1.1 : 1.0);
    return p;
}

// The key tiles (KT keys) that a query tile of 16 nw rows runs over: all, or its windows' span.
int spanned_tiles(const SdpaOptions& o, int n_tiles, int KT, int nw, int G) {
    return o.window > 0 ? (int)std::min<int64_t>(n_tiles, ((int64_t)o.window + 16 * nw / G + KT) / KT + 1)
                        : n_tiles;
}

RowsPlan choose_plan(int R, int G, int hkv, int n_tiles, int KT, const SdpaOptions& o) {
    RowsPlan p = plan_rows(R, hkv, 8, spanned_tiles(o, n_tiles, KT, 8, G));
    if (!o.mask) {
        const RowsPlan p12 = plan_rows(R, hkv, 12, spanned_tiles(o, n_tiles, KT, 12, G));
        if (p12.cost < p.cost) p = p12;
    }
    return p;
}

template <int D>
int rows_attention_d(const void* q, int G, int n_rows, const void* k, const void* v, int hkv,
                     int n_keys, int64_t khs, int64_t krs, int64_t vhs, int64_t vrs, float scale,
                     const SdpaOptions& o, void* out, hipStream_t stream) {
    using S = BlockShape<D>;
    const int R = G * n_rows, n_tiles = (n_keys + S::KT - 1) / S::KT;
    const RowsPlan p = choose_plan(R, G, hkv, n_tiles, S::KT, o);
    RowsArgs a;
    a.prow0 = p.q_main * 16 * p.nw;
    a.PR = R - a.prow0;
    // (the tiles below the first row's window are neither laid out nor read)
    const int tile0 = window_first_key(o, n_keys, n_rows, S::KT) / S::KT;
    const size_t img_bytes = (size_t)hkv * (n_tiles - tile0) * S::BUF;
    const size_t n_part = p.n_split > 1 ? (size_t)hkv * p.n_split * a.PR : 0;
    int dev = 0;
    QW_HIP_CHECK(hipGetDevice(&dev));
    void* ws = nullptr;
    if (int rc = workspace(kWsImages, dev, stream, img_bytes + n_part * (D * sizeof(float) + sizeof(float2)), &ws))
        return rc;
    a.q = (const f16*)q;
    a.out = (f16*)out;
    a.img = (const char*)ws;
    a.part_o = (float*)((char*)ws + img_bytes);
    a.part_ml = (float2*)(a.part_o + n_part * D);
    a.T = n_keys;
    a.Tq = n_rows;
    a.G = G;
    a.R = R;
    a.hkv = hkv;
    a.n_tiles = n_tiles;
    a.tile0 = tile0;
    a.causal = o.causal ? 1 : 0;
    a.window = o.window > 0 ? o.window : 0;
    a.n_main = p.q_main * hkv;
    a.qt0 = p.q_main;
    a.n_split = p.n_split;
    a.tiles_per_split = p.tps;
    a.mask = o.mask;
    a.mask_dtype = o.mask_dtype;
    a.mhs = o.mask_head_stride;
    a.mrs = o.mask_row_stride;
    a.scale_h = (float)(f16)scale;
    a.softcap = Softcap::of(scale, o.softcap);
    if (int rc = ensure_dynamic_lds((const void*)rows_image_kernel<D>, S::BUF)) return rc;
    hipLaunchKernelGGL((rows_image_kernel<D>), dim3(n_tiles - tile0, hkv), dim3(512), S::BUF,
                       stream, (const f16*)k, (const f16*)v, khs, krs, vhs, vrs, n_keys, tile0, (char*)ws);
    QW_HIP_CHECK(hipGetLastError());
    const int grid = a.n_main + (p.n_qt - p.q_main) * hkv * p.n_split;
    const bool cap = o.softcap > 0.0f;
    int rc;
    if (o.mask)
        rc = cap ? launch_rows_one<D, 8, true, true>(a, grid, stream)
                 : launch_rows_one<D, 8, false, true>(a, grid, stream);
    else if (p.nw == 8)
        rc = cap ? launch_rows_one<D, 8, true, false>(a, grid, stream)
                 : launch_rows_one<D, 8, false, false>(a, grid, stream);
    else
        rc = cap ? launch_rows_one<D, 12, true, false>(a, grid, stream)
                 : launch_rows_one<D, 12, false, false>(a, grid, stream);
    if (rc || p.n_split == 1) return rc;
    return launch_partial_merge(a.part_o, a.part_ml, p.n_split, a.PR, a.prow0, a.PR, hkv, D, G,
                                n_rows, (f16*)out, stream, 16);
}

}  // namespace

double rows_attention_us(int G, int n_rows, int hkv, int n_keys, int D, const SdpaOptions& o) {
    const int KT = 16384 / D, R = G * n_rows, n_tiles = (n_keys + KT - 1) / KT;
    const RowsPlan p = choose_plan(R, G, hkv, n_tiles, KT, o);
    const int PR = R - p.q_main * 16 * p.nw, tail = (p.n_qt - p.q_main) * hkv;
    const int tile0 = window_first_key(o, n_keys, n_rows, KT) / KT;
    // the longest run of key tiles on a CU
    const double cut = o.causal && o.window <= 0 ? 1.0 - 0.5 * n_rows / n_keys : 1.0;
    double chain = p.q_main * hkv / 256 * spanned_tiles(o, n_tiles, KT, p.nw, G) * cut;
    if (tail > 0) chain += (tail * p.n_split + 255) / 256 * p.tps;
    const double laid_out = 1e-6 * (n_tiles - tile0) * hkv * 16384;
    const double partials = p.n_split > 1 ? 8e-6 * p.n_split * hkv * PR * D : 0.0;  // MB
    double step = 1.9 + 80.0 / D;
    if (o.softcap > 0.0f) step += 0.2 + 150.0 / D;
    if (o.mask) step += (o.mask_dtype == QW_MASK_BOOL ? 130.0 : 280.0) / D;
    if (p.nw == 12) step *= 1.3;
    return 11.5 + 1.3 * laid_out + step * chain + (0.15 + 24.0 / D) * partials;
}

int rows_attention(const void* q, int G, int n_rows, const void* k, const void* v, int hkv,
                   int n_keys, int head_dim, int64_t khs, int64_t krs, int64_t vhs, int64_t vrs,
                   float scale, const SdpaOptions& o, void* out, hipStream_t stream) {
    if (head_dim == 256)
        return rows_attention_d<256>(q, G, n_rows, k, v, hkv, n_keys, khs, krs, vhs, vrs, scale, o, out, stream);
    if (head_dim == 128)
        return rows_attention_d<128>(q, G, n_rows, k, v, hkv, n_keys, khs, krs, vhs, vrs, scale, o, out, stream);
    return rows_attention_d<64>(q, G, n_rows, k, v, hkv, n_keys, khs, krs, vhs, vrs, scale, o, out, stream);
}

}  // namespace qw
