// dlsa_rows.hip - the D-LSA gathered read (K2) for prefill row counts, gfx950:
// neighbouring rows read the keys that any of them lists once.
//
// Contract: dlsa.hip's (the reference's dlsa_attention::sparse_attention,
// crates/mlxcel-core/src/dlsa_attention.rs:31-63): row r attends over the keys
// of its own list, entries outside [0, T) skipped, fp32 scores, softmax and sums,
// a row without a valid entry zeros. fp16 or bf16 q, K and V (alike) in those
// types; other pairs of types, and D = 32, in fp32 (dlsa_rows32_kernel).
//
// The rows of a prefill chunk list nearly the same keys (the sinks, the chunk's
// long-range blocks, windows that slide by one), but one row fills 6 of an MFMA
// tile's 16 columns and gathering its keys alone moves them once a row: 29 GB of
// L1 / L2 traffic for 1536 rows of 4612 keys. Here
//   dlsa_plan_kernel, one workgroup a group of NR neighbouring rows (NR G <= 128),
//     marks every listed key in an LDS bitmap word (bit i: row i of the group) and
//     compacts the marked keys in ascending order, with their words;
//   dlsa_rows_kernel, a workgroup a (group, KV head) as the block kernels have it:
//     128 columns (row, head), 64-key tiles gathered by the key list into the LDS
//     layout of block_tile.hpp, and for each score the key's bit of its row;
//   dlsa_rows_merge_kernel sums the fp32 partials of the groups whose keys were
//     split (the last, partial round of workgroups).
// P enters P.V as a high part plus a remainder in fp16, as in dlsa.hip, and in three
// parts in bf16, which hold the 24 bits of the fp32 P of dlsa_typed.hip (two hold 16:
// 512 rows at 16k 156 for 175 us, and an error against 64 bits of 1.655198e-3 for
// 1.655196e-3 here and there).
// What bounds it: MFMAs and LDS operand reads, as in attend_rows.hip, with three (bf16
// four) MFMAs a (key, column, dim) where that kernel has two. Measured (24 heads over 4,
// D = 256, lists of 4 sinks, a 512-key window and 8 shared 512-key blocks): 1536 rows
// at 32k in fp16 1312 us by row pairs -> 347 us here (502 TFLOP/s; the plan 26 us, the
// merge 6 us of it), 512 rows at 16k in bf16 7572 -> 175 us; in f32 7530 -> 744 us.
//
// A group is left to the row-by-row kernels, launched behind with the flags of
// this one, where (a) a row lists a key twice (it counts twice), (b) the union is
// larger than max_union (the rows share too little), or (c) an output came out
// infinite or NaN: a key's V reaches every row of its group here with weight 0,
// and 0 x inf is NaN.
#include <algorithm>

#include "block_tile.hpp"
#include "kv_cache.hpp"
#include "qw_common.hpp"

namespace qw {

namespace {

typedef __bf16 bhalf8 __attribute__((ext_vector_type(8)));
typedef uint16_t ushort4v __attribute__((ext_vector_type(4)));
typedef uint16_t ushort8v __attribute__((ext_vector_type(8)));

constexpr int kPlanSeg = 40448;  // keys a bitmap pass covers (158 KB of LDS)
constexpr int kPlanThreads = 1024;

// flags[group][hkv], nonzero for the row-by-row kernel: kLeft before the merge (by the
// plan, or by the row kernel for all groups together), kBad where an output came out
// infinite or NaN. No launch decides by a value that it writes: the row kernel reads
// the plan's counts alone, the merge only whether a flag is kLeft.
constexpr int kLeft = 1, kBad = 2;
__device__ __forceinline__ void set_flag(int* f, int value) {
    __hip_atomic_store(f, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool was_left(const int* f) {
    return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == kLeft;
}

// Group blockIdx.x: rows NR * blockIdx.x .. +NR-1. Writes its keys (ascending,
// padded with (0, no rows) to whole tiles of KT), their row words and the count;
// count -1 and flags[group][hkv] = kLeft if the group is not served.
__global__ __launch_bounds__(kPlanThreads) void dlsa_plan_kernel(
    const int32_t* __restrict__ lists, const int32_t* __restrict__ lengths, int L, int W, int T,
    int NR, int KT, int max_union, int cap, int hkv, int32_t* __restrict__ keys,
    uint32_t* __restrict__ words, int* __restrict__ counts, int* __restrict__ flags) {
    constexpr int NWV = kPlanThreads / 64;
    extern __shared__ __attribute__((aligned(16))) uint32_t bm[];  // min(T, kPlanSeg) words, whole u32x4
    __shared__ int wave_n[NWV];
    __shared__ int listed, marked;  // valid entries of the group's lists / bits set for them
    const int grp = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r0 = grp * NR, nr = min(NR, L - r0), n_chunks = (W + 255) / 256;
    int32_t* const gk = keys + (int64_t)grp * cap;
    uint32_t* const gw = words + (int64_t)grp * cap;
    if (tid == 0) listed = marked = 0;
    const int my_len = lane < nr ? min(lengths[r0 + lane], W) : 0;  // lane i: row i's length
    int total = 0, n_listed = 0, n_marked = 0;
    for (int seg = 0; seg < T; seg += kPlanSeg) {
        const int n = min(kPlanSeg, T - seg), n4 = (n + 3) / 4;
        __syncthreads();  // the previous segment's words are read
        for (int i = tid; i < n4; i += kPlanThreads) ((u32x4*)bm)[i] = u32x4{0, 0, 0, 0};
        __syncthreads();
        // 256-entry chunks of the lists (four entries a lane), dealt to the waves in
        // turn, eight of a wave in flight before the first is marked: a few
        // workgroups read all the lists from HBM (an entry a lane at a time, its
        // mark's old value awaited: 94 us for 1536 rows of 4612 entries)
        int r = 0, c = wave;  // the wave's next chunk: chunk c of row r
        auto next = [&]() {
            while (c >= n_chunks && r < nr) {
                c -= n_chunks;
                r++;
            }
        };
        next();
        while (r < nr) {
            constexpr int AH = 8;
            u32x4 x[AH];
            int row[AH];
#pragma unroll
            for (int i = 0; i < AH; i++) {
                row[i] = min(r, nr - 1);
                const int e = 256 * c + 4 * lane;
                const int left = r < nr ? __builtin_amdgcn_readlane(my_len, row[i]) - e : 0;
                const int32_t* p = lists + (int64_t)(r0 + row[i]) * W + e;
                x[i] = u32x4{~0u, ~0u, ~0u, ~0u};
                if (left >= 4) {
                    __builtin_memcpy(&x[i], p, 16);  // (rows are 4-byte aligned)
                } else {
#pragma unroll
                    for (int j = 0; j < 3; j++)
                        if (j < left) x[i][j] = (uint32_t)p[j];
                }
                c += NWV;
                next();
            }
#pragma unroll
            for (int i = 0; i < AH; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t key = x[i][j] - (uint32_t)seg;  // (below seg: wraps past n)
                    if ((int)x[i][j] >= 0 && key < (uint32_t)n) {
                        atomicOr(&bm[key], 1u << row[i]);
                        n_listed++;
                    }
                }
        }
        __syncthreads();
        // a wave's share in steps of 256 keys, four a lane: counted, then placed
        const int share = (n4 + 64 * NWV - 1) / (64 * NWV) * 64;  // (in quads)
        const int i0 = min(n4, wave * share), i1 = min(n4, i0 + share);
        auto quad = [&](int i) {
            return i + lane < i1 ? ((const u32x4*)bm)[i + lane] : u32x4{0, 0, 0, 0};
        };
        int cnt = 0;
        for (int i = i0; i < i1; i += 64) {
            const u32x4 w = quad(i);
            cnt += (w.x != 0) + (w.y != 0) + (w.z != 0) + (w.w != 0);
            n_marked += __popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w);
        }
        for (int x = 1; x < 64; x <<= 1) cnt += __shfl_xor(cnt, x);
        if (lane == 0) wave_n[wave] = cnt;
        __syncthreads();
        int pos = total;
        for (int w = 0; w < NWV; w++) {
            if (w < wave) pos += wave_n[w];
            total += wave_n[w];
        }
        for (int i = i0; i < i1; i += 64) {
            const u32x4 w = quad(i);
            const int c = (w.x != 0) + (w.y != 0) + (w.z != 0) + (w.w != 0);
            const uint64_t b0 = __ballot(c & 1), b1 = __ballot(c & 2), b2 = __ballot(c & 4);
            const uint64_t lt = (1ull << lane) - 1;
            int p = pos + __popcll(b0 & lt) + 2 * __popcll(b1 & lt) + 4 * __popcll(b2 & lt);
            pos += __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2);
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (w[j] != 0) {
                    if (p < cap) {
                        gk[p] = seg + 4 * (i + lane) + j;
                        gw[p] = w[j];
                    }
                    p++;
                }
        }
    }
    // a key that a row lists twice set one bit for two entries
    if (n_listed) atomicAdd(&listed, n_listed);
    if (n_marked) atomicAdd(&marked, n_marked);
    __syncthreads();
    const bool bad = listed != marked || total > max_union;
    if (!bad) {
        const int padded = (total + KT - 1) / KT * KT;  // <= cap
        for (int i = total + tid; i < padded; i += kPlanThreads) {
            gk[i] = 0;
            gw[i] = 0;
        }
    }
    if (tid == 0) counts[grp] = bad ? -1 : total;
    for (int h = tid; h < hkv; h += kPlanThreads) flags[grp * hkv + h] = bad ? kLeft : 0;
}

struct DlsaRowsArgs {
    const void* q;  // [hq][L][D]
    const void* k;  // element (h, t, d) at h * khs + t * krs + d
    const void* v;
    int64_t khs, krs, vhs, vrs;
    void* out;       // [hq][L][D]
    float* part_o;   // [hkv][n_split][PR][D] in V slot order, rows from prow0
    float2* part_ml; // [hkv][n_split][PR] (m in log2 units)
    const int32_t* keys;    // [groups][cap]
    const uint32_t* words;
    const int* counts;      // [groups] (the plan's, -1: not served)
    int* flags;             // [groups][hkv], see kLeft
    int L, G, hkv, NR, cap, groups;
    int n_main, qt0, n_split, prow0, PR;  // as RowsArgs (attend_rows.hip)
    float scale2;           // scale * log2(e)
    int q_dtype;            // q's and out's type (the fp32 kernel)
};

template <bool BF>
struct Elem;
template <>
struct Elem<false> {
    typedef half8 V8;
    __device__ static float4v mfma(V8 a, V8 b, float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    typedef f16 T;
};
template <>
struct Elem<true> {
    typedef bhalf8 V8;
    __device__ static float4v mfma(V8 a, V8 b, float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    typedef __bf16 T;
};

__device__ __forceinline__ void store_as(void* out, int dtype, int64_t at, float y) {
    if (dtype == QW_DTYPE_F32) ((float*)out)[at] = y;
    else if (dtype == QW_DTYPE_F16) ((f16*)out)[at] = (f16)y;
    else ((__bf16*)out)[at] = (__bf16)y;
}

// Whether group qt goes to the row-by-row kernel, for all 512 threads (the launch writes no
// count): by the plan, or because more than a quarter of the groups do. Both launches are
// then long however few groups each has, and a mixture costs their sum: fp16, 512 rows of
// which half share too little, 649 us, 364 by rows alone; f32, 24 heads over 3, D = 128, 1100
// rows of which the last 12 would be served, 1038 us, 608 by rows alone.
__device__ __forceinline__ bool group_left(const DlsaRowsArgs& a, int qt, int h) {
    if (a.counts[qt] < 0) return true;
    int left = 0;
    for (int i = 0; i < a.groups; i += 512)
        left += __syncthreads_count(i + (int)threadIdx.x < a.groups && a.counts[i + threadIdx.x] < 0);
    if (4 * left <= a.groups) return false;
    if (threadIdx.x == 0) set_flag(a.flags + qt * a.hkv + h, kLeft);
    return true;
}

template <int D, bool BF>
__global__ __launch_bounds__(512, 1) void dlsa_rows_kernel(DlsaRowsArgs a) {
    using S = BlockShape<D>;
    using E = Elem<BF>;
    using V8 = typename E::V8;
    using ET = typename E::T;
    constexpr int KT = S::KT, NSUB = S::NSUB, NM = S::NM, NT = S::NT, BUF = S::BUF, KBUF = S::KBUF;
    constexpr int VROW = S::VROW, TPR = S::TPR, TPB = S::TPB;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint32_t* const sW = (uint32_t*)(lds + 2 * BUF);  // [2][KT] row words
    int sp = 0, qt, h, n_split = 1;
    {
        const int lin = blockIdx.x;
        if (lin < a.n_main) {
            qt = lin / a.hkv;
            h = lin % a.hkv;
        } else {
            const int t = lin - a.n_main;
            n_split = a.n_split;
            sp = t % n_split;
            h = (t / n_split) % a.hkv;
            qt = a.qt0 + t / (n_split * a.hkv);
        }
    }
    if (group_left(a, qt, h)) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int n_tiles = (a.counts[qt] + KT - 1) / KT, tps = (n_tiles + n_split - 1) / n_split;
    const int t0 = sp * tps, t1 = min(n_tiles, t0 + tps);
    // columns: (row of the group, head), row * G + head
    const int R = a.L * a.G, row0 = qt * a.NR * a.G, row_end = min(R, row0 + a.NR * a.G);
    const int wrow0 = row0 + 16 * wave, rho = wrow0 + r16;
    const bool wave_live = wrow0 < row_end, row_ok = rho < row_end;
    const int r = row_ok ? rho / a.G : 0, qh = h * a.G + (row_ok ? rho - r * a.G : 0);
    const int bit = row_ok ? r - qt * a.NR : 0;  // the column's row in the words
    // the rows of the wave's columns
    const int b_lo = wave_live ? (wrow0 - row0) / a.G : 0;
    const int b_hi = wave_live ? (min(row_end, wrow0 + 16) - 1 - row0) / a.G : 0;
    const uint32_t need = (b_hi - b_lo == 31 ? ~0u : ((1u << (b_hi - b_lo + 1)) - 1)) << b_lo;

    V8 qb[NM];
    {
        const ET* qrow = (const ET*)a.q + ((int64_t)qh * a.L + r) * D;
#pragma unroll
        for (int m = 0; m < NM; m++) qb[m] = *(const V8*)(qrow + 32 * m + 8 * g);
    }

    // tile loads: the 32-dim slice q32 of key kk of K, and 4 dims from 4 vj of
    // the 8 keys of block vb of V (64 lanes read whole rows); the keys of the
    // tile after the one being loaded are already in registers
    static_assert(KT * TPR == 512 && (KT / 8) * TPB == 512, "one slice of each kind a thread");
    const int q32 = (tid >> 4) & (TPR - 1), kk = (tid & 15) | ((tid >> (4 + S::LTPR)) << 4);
    const int vb = tid / TPB, vj = tid % TPB;
    const uint16_t* const kh = (const uint16_t*)a.k + h * a.khs + 32 * q32;
    const uint16_t* const vh = (const uint16_t*)a.v + h * a.vhs + 4 * vj;
    const int32_t* const gk = a.keys + (int64_t)qt * a.cap;
    const uint32_t* const gw = a.words + (int64_t)qt * a.cap;
    int ki, vi[8];
    auto index = [&](int t) {
        ki = gk[t * KT + kk];
        const int32_t* p = gk + t * KT + 8 * vb;
#pragma unroll
        for (int i = 0; i < 8; i++) vi[i] = p[i];
    };
    u32x4 kc[4];
    ushort4v vr[8];
    uint32_t word;
    auto load = [&](int t) {
        const u32x4* ks = (const u32x4*)(kh + ki * a.krs);
#pragma unroll
        for (int w = 0; w < 4; w++) kc[w] = ks[w];
#pragma unroll
        for (int i = 0; i < 8; i++) vr[i] = *(const ushort4v*)(vh + vi[i] * a.vrs);
        if (tid < KT) word = gw[t * KT + tid];
    };
    auto store = [&](int b) {
        u32x4* const sK = (u32x4*)(lds + BUF * b) + kaddr<KT>(kk, 4 * q32);
        ushort8v* const sV = (ushort8v*)(lds + BUF * b + KBUF) + vb * VROW;
#pragma unroll
        for (int w = 0; w < 4; w++) sK[w * KT] = kc[w];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            ushort8v y;
#pragma unroll
            for (int i = 0; i < 8; i++) y[i] = vr[i][e];
            const int sl = v_phys_dim(4 * vj + e, D, 16);
            sV[sl + (sl >> 4)] = y;
        }
        if (tid < KT) sW[b * KT + tid] = word;
    };

    float m_run = -INFINITY, l_run = 0.0f;
    float4v acc_o[NT];
#pragma unroll
    for (int mm = 0; mm < NT; mm++) acc_o[mm] = float4v{0.f, 0.f, 0.f, 0.f};

    // NU 32-key sub-blocks from sub-block ub of buffer b
    constexpr int NU = NSUB < 4 ? NSUB : 4;
    auto tile = [&](int b, int ub) {
        const V8* sK8 = (const V8*)(lds + BUF * b) + 32 * ub;
        const V8* sV8 = (const V8*)(lds + BUF * b + KBUF) + 4 * ub * VROW;
        // the lane's keys 32u + 8g + e
        uint32_t w[NU][8], all = ~0u, any = 0;
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const u32x4* p = (const u32x4*)(sW + b * KT + 32 * (ub + u) + 8 * g);
            const u32x4 x = p[0], y = p[1];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                w[u][e] = e < 4 ? x[e & 3] : y[e & 3];
                all &= w[u][e];
                any |= w[u][e];
            }
        }
        if (!__any((any & need) != 0)) return;  // none of the wave's rows lists any of them
        const bool full = __all((all & need) == need);
        const int key0 = 8 * (r16 >> 2) + (r16 & 3);
        const int b4 = (key0 >> 4) & 1;
        const V8* kbase0 = sK8 + g * KT + key0 + 4 * b4;
        const V8* kbase1 = sK8 + g * KT + key0 + 4 * (b4 ^ 1);
        float4v acc[NU][2];
#pragma unroll
        for (int u = 0; u < NU; u++) acc[u][0] = acc[u][1] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const V8 ka = kbase0[4 * m * KT + 32 * u], kb2 = kbase1[4 * m * KT + 32 * u];
                acc[u][0] = E::mfma(ka, qb[m], acc[u][0]);
                acc[u][1] = E::mfma(kb2, qb[m], acc[u][1]);
            }
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
        float sf[NU][8];
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int e = 0; e < 8; e++) sf[u][e] = acc[u][e >> 2][e & 3] * a.scale2;
        if (!full) {
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (((w[u][e] >> bit) & 1u) == 0) sf[u][e] = -INFINITY;
        }
        float mx = sf[0][0];
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int e = 0; e < 8; e++) mx = fmaxf(mx, sf[u][e]);
        // lazy reference in log2 units (p <= 2^5.5)
        if (__any(mx > m_run + 5.5f)) {
            const float m_new = fmaxf(m_run, wave_max_g(mx));
            if (__any(m_run != -INFINITY)) {
                const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
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
        const float mref = m_run == -INFINITY ? 0.0f : m_run;
        V8 ph[NU], pl[NU], pm[BF ? NU : 1];
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float p = __builtin_amdgcn_exp2f(sf[u][e] - mref);
                l_run += p;
                ph[u][e] = (ET)p;
                const float rest = p - (float)ph[u][e];
                pl[u][e] = (ET)rest;
                if constexpr (BF) pm[u][e] = (ET)(rest - (float)pl[u][e]);
            }
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const V8* vb8 = sV8 + (4 * u + g) * VROW + r16;
#pragma unroll
            for (int mm = 0; mm < NT; mm++) {
                const V8 vv = vb8[17 * mm];
                acc_o[mm] = E::mfma(ph[u], vv, acc_o[mm]);
                acc_o[mm] = E::mfma(pl[u], vv, acc_o[mm]);
                if constexpr (BF) acc_o[mm] = E::mfma(pm[u], vv, acc_o[mm]);
            }
        }
        {
            constexpr int NQ = NU * NT, AH = 4, MF = BF ? 3 : 2;
            __builtin_amdgcn_sched_group_barrier(0x100, AH, 1);
#pragma unroll
            for (int i = 0; i < NQ - AH; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, MF, 1);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, MF * AH, 1);
        }
    };

    // round t: tile t+1 (in registers) into the free buffer, the loads of tile
    // t+2 and the key indexes of tile t+3, tile t's math; one barrier
    if (t0 < t1) {
        index(t0);
        load(t0);
        if (t0 + 1 < t1) index(t0 + 1);
        store(0);
        if (t0 + 1 < t1) load(t0 + 1);
        if (t0 + 2 < t1) index(t0 + 2);
    }
    __syncthreads();
    for (int t = t0; t < t1; t++) {
        const int b = (t - t0) & 1;
        if (t + 1 < t1) {
            store(b ^ 1);
            if (t + 2 < t1) load(t + 2);
            if (t + 3 < t1) index(t + 3);
        }
        if (wave_live) {
#pragma unroll
            for (int ub = 0; ub < NSUB; ub += NU) tile(b, ub);
        }
        __syncthreads();
    }

    const float lsum = wave_sum_g(l_run);
    if (n_split == 1) {
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float l = __shfl(lsum, 4 * g + i);
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            const int row = wrow0 + 4 * g + i;
            if (row >= row_end) continue;
            ET* orow = (ET*)a.out + ((int64_t)(h * a.G + row % a.G) * a.L + row / a.G) * D;
            // slot 16mm + r16 is dim NT r16 + mm: a lane's NT dims are consecutive
#pragma unroll
            for (int mm = 0; mm < NT; mm++) {
                const float o = acc_o[mm][i] * inv;
                bad |= !(fabsf(o) < INFINITY);
                orow[NT * r16 + mm] = (ET)o;
            }
            bad |= !(fabsf(l) < INFINITY);
        }
        if (bad) set_flag(a.flags + qt * a.hkv + h, kBad);
    } else {
        const int64_t pbase = ((int64_t)h * n_split + sp) * a.PR - a.prow0;
        if (g == 0 && row_ok) a.part_ml[pbase + rho] = float2{m_run, lsum};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = wrow0 + 4 * g + i;
            if (row >= row_end) continue;
            float* prow = a.part_o + (pbase + row) * D;
#pragma unroll
            for (int mm = 0; mm < NT; mm++) prow[16 * mm + r16] = acc_o[mm][i];
        }
    }
}

// out row = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s over the splits, in the
// element type. grid (rows of the split groups / 4, KV heads), a wave a row, a lane
// D / 64 consecutive slots, the partials loaded four at a time.
template <int D, bool BF>
__global__ __launch_bounds__(256) void dlsa_rows_merge_kernel(DlsaRowsArgs a) {
    using ET = typename Elem<BF>::T;
    constexpr int SPL = D / 64;
    typedef float vec __attribute__((ext_vector_type(SPL)));
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int pr = blockIdx.x * 4 + wave, h = blockIdx.y;
    if (pr >= a.PR) return;
    const int row = a.prow0 + pr, grp = row / (a.NR * a.G), fl = grp * a.hkv + h;
    if (was_left(a.flags + fl)) return;
    const int64_t base = (int64_t)h * a.n_split * a.PR + pr;
    float M = -INFINITY, l = 0.0f;
    vec o = {};
    for (int c0 = 0; c0 < a.n_split; c0 += 4) {
        float2 ml[4];
        vec x[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t at = base + (int64_t)min(c0 + i, a.n_split - 1) * a.PR;
            ml[i] = a.part_ml[at];
            x[i] = *(const vec*)(a.part_o + at * D + SPL * lane);
            if (c0 + i >= a.n_split) ml[i] = float2{-INFINITY, 0.0f};
        }
        float m = M;
#pragma unroll
        for (int i = 0; i < 4; i++) m = fmaxf(m, ml[i].x);
        if (m == -INFINITY) continue;
        const float f0 = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - m);
        o = o * f0;
        l *= f0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float f = ml[i].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[i].x - m);
            o += f * x[i];
            l = __builtin_fmaf(f, ml[i].y, l);
        }
        M = m;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const int r = row / a.G, qh = h * a.G + row % a.G;
    ET* const orow = (ET*)a.out + ((int64_t)qh * a.L + r) * D;
    bool bad = !(fabsf(l) < INFINITY);
#pragma unroll
    for (int j = 0; j < SPL; j++) {
        const float y = o[j] * inv;
        bad |= !(fabsf(y) < INFINITY);
        orow[v_logical_dim(SPL * lane + j, D, 16)] = (ET)y;
    }
    if (bad) set_flag(a.flags + fl, kBad);
}

// The same in fp32 throughout, for every other pair of types (and D = 32): K and V
// rows widened to fp32 as they are staged, both products on
// v_mfma_f32_16x16x4_f32. Bound by those MFMAs (a sixteenth of the 16-bit rate).
// Layouts: tiles of 8192 / D keys; the four MFMAs of a 16-dim chunk take element
// 0 .. 3 of each lane's 16-byte piece (lane (g, r16): dims 16m + 4g .. +3), so K is
// read 16 bytes a lane, chunk c of key k at c ^ (k mod 16) against bank conflicts; P
// leaves the score tile as the A operand (keys 4g + i, MFMA i), and V is read VD dims
// a lane of one key, one operand for each of VD output tiles.
template <int D, int DKV>
__global__ __launch_bounds__(512, 1) void dlsa_rows32_kernel(DlsaRowsArgs a) {
    constexpr int KT = 8192 / D, CPR = D / 4;  // keys a tile, 16-byte chunks a row
    constexpr int NM = D / 16, SW = CPR < 16 ? CPR - 1 : 15;
    constexpr int VD = D < 64 ? 2 : 4, NP = D / (16 * VD);
    constexpr int KBUF = KT * D * 4;  // bytes of a K (V) tile: 32 KB
    constexpr int WPT = DKV == QW_DTYPE_F32 ? 4 : 2;  // 16-byte pieces of 16 values
    typedef float vecv __attribute__((ext_vector_type(VD)));
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint32_t* const sW = (uint32_t*)(lds + 4 * KBUF);  // [2][KT] row words
    int sp = 0, qt, h, n_split = 1;
    {
        const int lin = blockIdx.x;
        if (lin < a.n_main) {
            qt = lin / a.hkv;
            h = lin % a.hkv;
        } else {
            const int t = lin - a.n_main;
            n_split = a.n_split;
            sp = t % n_split;
            h = (t / n_split) % a.hkv;
            qt = a.qt0 + t / (n_split * a.hkv);
        }
    }
    if (group_left(a, qt, h)) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int n_tiles = (a.counts[qt] + KT - 1) / KT, tps = (n_tiles + n_split - 1) / n_split;
    const int t0 = sp * tps, t1 = min(n_tiles, t0 + tps);
    const int R = a.L * a.G, row0 = qt * a.NR * a.G, row_end = min(R, row0 + a.NR * a.G);
    const int wrow0 = row0 + 16 * wave, rho = wrow0 + r16;
    const bool wave_live = wrow0 < row_end, row_ok = rho < row_end;
    const int r = row_ok ? rho / a.G : 0, qh = h * a.G + (row_ok ? rho - r * a.G : 0);
    const int bit = row_ok ? r - qt * a.NR : 0;
    float4v qb[NM];
    {
        const int64_t q0 = ((int64_t)qh * a.L + r) * D;
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int64_t at = q0 + 16 * m + 4 * g + e;
                qb[m][e] = a.q_dtype == QW_DTYPE_F32   ? ((const float*)a.q)[at]
                           : a.q_dtype == QW_DTYPE_F16 ? (float)((const f16*)a.q)[at]
                                                       : (float)((const __bf16*)a.q)[at];
            }
    }
    // a thread stages 16 dims of one key, of K and of V
    const int kk = tid / (D / 16), sl = tid % (D / 16);
    constexpr int ES = DKV == QW_DTYPE_F32 ? 4 : 2;
    const char* const kh = (const char*)a.k + ES * (h * a.khs + 16 * sl);
    const char* const vh = (const char*)a.v + ES * (h * a.vhs + 16 * sl);
    const int32_t* const gk = a.keys + (int64_t)qt * a.cap;
    const uint32_t* const gw = a.words + (int64_t)qt * a.cap;
    int ki;
    u32x4 kc[WPT], vc[WPT];
    uint32_t word;
    auto load = [&](int t) {
        const u32x4* ks = (const u32x4*)(kh + ES * ki * a.krs);
        const u32x4* vs = (const u32x4*)(vh + ES * ki * a.vrs);
#pragma unroll
        for (int w = 0; w < WPT; w++) {
            kc[w] = ks[w];
            vc[w] = vs[w];
        }
        if (tid < KT) word = gw[t * KT + tid];
    };
    auto wide = [&](const u32x4* c, int w) {  // values 4w .. 4w + 3
        if constexpr (DKV == QW_DTYPE_F32) {
            return __builtin_bit_cast(float4v, c[w]);
        } else {
            const uint32_t x = c[w / 2][2 * (w & 1)], y = c[w / 2][2 * (w & 1) + 1];
            if constexpr (DKV == QW_DTYPE_F16)
                return float4v{(float)h2(x).x, (float)h2(x).y, (float)h2(y).x, (float)h2(y).y};
            else
                return float4v{__uint_as_float(x << 16), __uint_as_float(x & 0xFFFF0000u),
                               __uint_as_float(y << 16), __uint_as_float(y & 0xFFFF0000u)};
        }
    };
    auto store = [&](int b) {
        float4v* const sK = (float4v*)(lds + 2 * KBUF * b) + kk * CPR;
        float4v* const sV = (float4v*)(lds + 2 * KBUF * b + KBUF) + kk * CPR;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            sK[(4 * sl + w) ^ (kk & SW)] = wide(kc, w);
            sV[4 * sl + w] = wide(vc, w);
        }
        if (tid < KT) sW[b * KT + tid] = word;
    };

    float m_run = -INFINITY, l_run = 0.0f;
    float4v acc_o[NP][VD];
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
        for (int c = 0; c < VD; c++) acc_o[p][c] = float4v{0.f, 0.f, 0.f, 0.f};

    // 16 keys from key k0 of buffer b: lane (g, r16) has keys 4g + i of column r16
    auto tile = [&](int b, int k0) {
        const float4v* const sK = (const float4v*)(lds + 2 * KBUF * b) + (k0 + r16) * CPR;
        const float* const sV = (const float*)(lds + 2 * KBUF * b + KBUF) + (k0 + 4 * g) * D + VD * r16;
        const u32x4 w4 = *(const u32x4*)(sW + b * KT + k0 + 4 * g);
        if (!__any(row_ok && (((w4.x | w4.y | w4.z | w4.w) >> bit) & 1u))) return;
        float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const float4v ka = sK[(4 * m + g) ^ (r16 & SW)];
#pragma unroll
            for (int e = 0; e < 4; e++)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[e], qb[m][e], acc, 0, 0, 0);
        }
        float sf[4];
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sf[i] = (w4[i] >> bit) & 1u ? acc[i] * a.scale2 : -INFINITY;
            mx = fmaxf(mx, sf[i]);
        }
        if (__any(mx > m_run + 5.5f)) {
            const float m_new = fmaxf(m_run, wave_max_g(mx));
            if (__any(m_run != -INFINITY)) {
                const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
                l_run *= alpha;
                float f[4];
#pragma unroll
                for (int i = 0; i < 4; i++) f[i] = __shfl(alpha, 4 * g + i);
#pragma unroll
                for (int p = 0; p < NP; p++)
#pragma unroll
                    for (int c = 0; c < VD; c++)
#pragma unroll
                        for (int i = 0; i < 4; i++) acc_o[p][c][i] *= f[i];
            }
            m_run = m_new;
        }
        const float mref = m_run == -INFINITY ? 0.0f : m_run;
        float pr[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            pr[i] = __builtin_amdgcn_exp2f(sf[i] - mref);
            l_run += pr[i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int p = 0; p < NP; p++) {
                const vecv vv = *(const vecv*)(sV + i * D + 16 * VD * p);
#pragma unroll
                for (int c = 0; c < VD; c++)
                    acc_o[p][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(pr[i], vv[c], acc_o[p][c], 0, 0, 0);
            }
    };

    if (t0 < t1) {
        ki = gk[t0 * KT + kk];
        load(t0);
        if (t0 + 1 < t1) ki = gk[(t0 + 1) * KT + kk];
        store(0);
        if (t0 + 1 < t1) load(t0 + 1);
        if (t0 + 2 < t1) ki = gk[(t0 + 2) * KT + kk];
    }
    __syncthreads();
    for (int t = t0; t < t1; t++) {
        const int b = (t - t0) & 1;
        if (t + 1 < t1) {
            store(b ^ 1);
            if (t + 2 < t1) load(t + 2);
            if (t + 3 < t1) ki = gk[(t + 3) * KT + kk];
        }
        if (wave_live) {
#pragma unroll 2
            for (int k0 = 0; k0 < KT; k0 += 16) tile(b, k0);
        }
        __syncthreads();
    }

    // column 4g + i of the wave, dims 16 VD p + VD r16 + c
    const float lsum = wave_sum_g(l_run);
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float l = __shfl(lsum, 4 * g + i);
        const int row = wrow0 + 4 * g + i;
        if (row >= row_end) continue;
        if (n_split > 1) {
            float* prow = a.part_o + (((int64_t)h * n_split + sp) * a.PR - a.prow0 + row) * D;
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int c = 0; c < VD; c++) prow[16 * VD * p + VD * r16 + c] = acc_o[p][c][i];
            continue;
        }
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        bad |= !(fabsf(l) < INFINITY);
        const int64_t o0 = ((int64_t)(h * a.G + row % a.G) * a.L + row / a.G) * D;
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int c = 0; c < VD; c++) {
                const float y = acc_o[p][c][i] * inv;
                bad |= !(fabsf(y) < INFINITY);
                store_as(a.out, a.q_dtype, o0 + 16 * VD * p + VD * r16 + c, y);
            }
    }
    if (n_split > 1) {
        if (g == 0 && row_ok)
            a.part_ml[((int64_t)h * n_split + sp) * a.PR - a.prow0 + rho] = float2{m_run, lsum};
    } else if (bad) {
        set_flag(a.flags + qt * a.hkv + h, kBad);
    }
}

// Its merge: grid (rows of the split groups, KV heads), D threads (dims).
__global__ void dlsa_rows32_merge_kernel(DlsaRowsArgs a) {
    const int D = blockDim.x, d = threadIdx.x, pr = blockIdx.x, h = blockIdx.y;
    const int row = a.prow0 + pr, fl = row / (a.NR * a.G) * a.hkv + h;
    if (was_left(a.flags + fl)) return;
    const int64_t base = (int64_t)h * a.n_split * a.PR + pr;
    float M = -INFINITY, o = 0.0f, l = 0.0f;
    for (int c0 = 0; c0 < a.n_split; c0 += 4) {
        float2 ml[4];
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t at = base + (int64_t)min(c0 + i, a.n_split - 1) * a.PR;
            ml[i] = a.part_ml[at];
            x[i] = a.part_o[at * D + d];
            if (c0 + i >= a.n_split) ml[i] = float2{-INFINITY, 0.0f};
        }
        float m = M;
#pragma unroll
        for (int i = 0; i < 4; i++) m = fmaxf(m, ml[i].x);
        if (m == -INFINITY) continue;
        const float f0 = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - m);
        o *= f0;
        l *= f0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float f = ml[i].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[i].x - m);
            o = __builtin_fmaf(f, x[i], o);
            l = __builtin_fmaf(f, ml[i].y, l);
        }
        M = m;
    }
    const float y = l > 0.0f ? o / l : 0.0f;
    if (!(fabsf(y) < INFINITY) || !(fabsf(l) < INFINITY)) set_flag(a.flags + fl, kBad);
    store_as(a.out, a.q_dtype, ((int64_t)(h * a.G + row % a.G) * a.L + row / a.G) * D + d, y);
}

template <int D, bool BF>
int launch_rows(const DlsaRowsArgs& a, int grid, hipStream_t stream) {
    const size_t shmem = 2 * BlockShape<D>::BUF + 2 * BlockShape<D>::KT * sizeof(uint32_t);
    if (int rc = ensure_dynamic_lds((const void*)dlsa_rows_kernel<D, BF>, shmem)) return rc;
    hipLaunchKernelGGL((dlsa_rows_kernel<D, BF>), dim3(grid), dim3(512), shmem, stream, a);
    QW_HIP_CHECK(hipGetLastError());
    if (a.n_split > 1) {
        hipLaunchKernelGGL((dlsa_rows_merge_kernel<D, BF>), dim3((a.PR + 3) / 4, a.hkv), dim3(256), 0,
                           stream, a);
        QW_HIP_CHECK(hipGetLastError());
    }
    return QW_OK;
}

template <int D, int DKV>
int launch_rows32(const DlsaRowsArgs& a, int grid, hipStream_t stream) {
    const size_t shmem = (size_t)4 * 32768 + 2 * (8192 / D) * sizeof(uint32_t);
    if (int rc = ensure_dynamic_lds((const void*)dlsa_rows32_kernel<D, DKV>, shmem)) return rc;
    hipLaunchKernelGGL((dlsa_rows32_kernel<D, DKV>), dim3(grid), dim3(512), shmem, stream, a);
    QW_HIP_CHECK(hipGetLastError());
    if (a.n_split > 1) {
        hipLaunchKernelGGL(dlsa_rows32_merge_kernel, dim3(a.PR, a.hkv), dim3(D), 0, stream, a);
        QW_HIP_CHECK(hipGetLastError());
    }
    return QW_OK;
}

template <int DKV>
int launch_rows32(const DlsaRowsArgs& a, int D, int grid, hipStream_t stream) {
    switch (D) {
        case 32: return launch_rows32<32, DKV>(a, grid, stream);
        case 64: return launch_rows32<64, DKV>(a, grid, stream);
        case 128: return launch_rows32<128, DKV>(a, grid, stream);
        default: return launch_rows32<256, DKV>(a, grid, stream);
    }
}

}  // namespace

int dlsa_rows_per_group(int G) { return std::min(32, 128 / G) & ~1; }

// How the groups of a call are divided: whole rounds of unsplit workgroups, the rest split
// over their keys, at least four tiles of the largest union each (those past a smaller
// one's end cost a launch slot and an empty partial).
struct GroupPlan {
    int groups, q_main, n_split;  // groups in all, in whole rounds, and the splits of the rest
};
static GroupPlan plan_groups(int n_rows, int n_kv_heads, int NR, int64_t tiles) {
    GroupPlan p{(n_rows + NR - 1) / NR, 0, 1};
    const int64_t units = (int64_t)p.groups * n_kv_heads;
    if (units >= 256 && 256 % n_kv_heads == 0) p.q_main = (int)(units / 256) * (256 / n_kv_heads);
    const int64_t tail = (int64_t)(p.groups - p.q_main) * n_kv_heads;
    if (tail > 0) p.n_split = (int)std::max<int64_t>(1, std::min({256 / tail, tiles / 4, (int64_t)32}));
    return p;
}

// The largest union of a group that is worth serving here, 0 for a call that is not: where
// the time here, estimated from the plan, a cost of the launches and one a key of the
// unions, meets the estimate for the kernel that runs row by row behind (by row pairs in
// fp16, dlsa_typed.hip for the other types). A call is taken if it gains a tenth where the
// rows share nearly all keys, as a prefill chunk's do. The coefficients are fitted to 3,100
// calls timed by both (eight head geometries at D = 64 / 128 / 256, 64 to 4608 entries of 1k
// to 66k keys, 33 to 1100 rows; lists shared, sliding, drawn in blocks and singly): nine in
// ten estimates within 25 %.
// Here / by rows, lists shared and drawn singly, in us: fp16, 24 heads over 4, D = 256, 1536
// rows of 4612 entries 345 / 1312; 16 over 2, D = 64, 1100 rows of 1024 entries drawn singly
// from 4k keys 110 / 72 (left); bf16, 24 over 4, D = 256, 48 rows of 128 38 / 79; f32, 8 over 8, D =
// 128, 96 rows of 64 28 / 17 and 47 / 21 (left).
// Where a union may be larger than that, rows that share next to nothing pay the plan
// (some 16 us, and 0.45 a thousand keys) for nothing, and nothing on the host tells them
// from rows that share. A typed call is taken where that is at most a quarter of its
// time, an fp16 call from 12M entries of 256 dims over the heads, where it measured 2 to 5 %
// (D = 256, 8 heads, 329 rows 1613 -> 1676 us; D = 128, 32 over 8, 658 rows 1444 -> 1516).
int64_t dlsa_rows_union(int q_dtype, int kv_dtype, int n_rows, int width, int n_kv_heads, int G, int D,
                        int n_keys, hipStream_t stream) {
    if (stream == hipStreamPerThread) return 0;  // (one handle, a stream a thread)
    const bool alike = q_dtype == kv_dtype && kv_dtype != QW_DTYPE_F32 && D != 32;
    const bool pairs = alike && q_dtype == QW_DTYPE_F16;
    if (pairs && (n_rows < 32 || (int64_t)n_rows * n_kv_heads <= 256)) return 0;
    const int NR = dlsa_rows_per_group(G), KT = (alike ? 16384 : 8192) / D;
    const double W = width, entries = 1e-6 * n_rows * W * n_kv_heads, drawn = (double)NR * W;
    const double most = std::min<double>(n_keys, drawn), close = std::min<double>(n_keys, 1.3 * W + 2 * NR);
    // row by row: a list's own length in time, however few the rows, and the entries' share
    const double list = pairs ? 10 + 0.0085 * W : 9 + (0.045 + 0.06 * G) * W;
    const double rows = list + (pairs ? 3 + 0.215 * D : 62 + 0.13 * D + (31 + 0.125 * D) * G) * entries;
    const GroupPlan p = plan_groups(n_rows, n_kv_heads, NR, (int64_t)(most + KT - 1) / KT);
    const int64_t tail = (int64_t)(p.groups - p.q_main) * n_kv_heads;
    const double partials = p.n_split > 1 ? 8e-6 * p.n_split * n_kv_heads * D *
                                                ((double)n_rows * G - (double)p.q_main * NR * G)
                                          : 0.0;  // MB
    const double rounds = (double)p.q_main * n_kv_heads / 256 +
                          (tail > 0 ? (double)((tail * p.n_split + 255) / 256) / p.n_split : 0.0);
    const double tile = pairs ? 2.4 + 155.0 / D : alike ? 2.6 + 180.0 / D : 7.3;
    const double launches = (alike ? 21 : 24) + 0.45e-3 * n_keys + (0.12 + 35.0 / D) * partials;
    const double key = tile / KT * rounds;
    double limit = ((pairs ? 1.0 : 0.8) * rows - launches) / key;
    if (pairs) {
        limit = std::min(limit, 0.35 * drawn - 1500);
    } else if (limit < most) {
        // (a group that is left costs `list` beside the time here, so where some may be,
        // unions far above a list are served only if both together take less)
        limit = std::min(limit, std::max((rows - list - launches) / key, 1.1 * close));
    }
    if (limit <= close || (alike ? 1.1 : 1.3) * (launches + key * close) >= rows) return 0;
    if (limit < most && (pairs ? entries * D < 12.0 * 256 : 16 + 0.45e-3 * n_keys > 0.25 * rows)) return 0;
    return (int64_t)std::min(limit, most);
}

int dlsa_rows_attention(const void* q, int q_dtype, const void* k, const void* v, int kv_dtype,
                        int64_t khs, int64_t krs, int64_t vhs, int64_t vrs, const int32_t* lists,
                        const int32_t* lengths, int n_rows, int width, int n_q_heads,
                        int n_kv_heads, int D, int n_keys, int64_t most, float scale, void* out,
                        const int** flags, hipStream_t stream) {
    const int G = n_q_heads / n_kv_heads, NR = dlsa_rows_per_group(G);
    const bool fp16 = q_dtype == QW_DTYPE_F16 && kv_dtype == QW_DTYPE_F16;
    const bool bf16 = q_dtype == QW_DTYPE_BF16 && kv_dtype == QW_DTYPE_BF16;
    const bool rows32 = !(fp16 || bf16) || D == 32;
    const int KT = (rows32 ? 8192 : 16384) / D, max_union = (int)most;
    const int cap = (max_union + KT - 1) / KT * KT;
    const GroupPlan plan = plan_groups(n_rows, n_kv_heads, NR, cap / KT);
    const int groups = plan.groups, q_main = plan.q_main, units = groups * n_kv_heads;
    DlsaRowsArgs a;
    a.n_split = plan.n_split;
    a.n_main = q_main * n_kv_heads;
    a.qt0 = q_main;
    a.prow0 = q_main * NR * G;
    a.PR = n_rows * G - a.prow0;
    const size_t n_part = a.n_split > 1 ? (size_t)n_kv_heads * a.n_split * a.PR : 0;
    const size_t part_bytes = n_part * (D * sizeof(float) + sizeof(float2));
    const size_t list_bytes = (size_t)groups * cap * sizeof(int32_t);
    const size_t count_bytes = (size_t)(groups + 3) / 4 * 4 * sizeof(int);
    int dev = 0;
    QW_HIP_CHECK(hipGetDevice(&dev));
    void* ws = nullptr;
    if (int rc = workspace(kWsUnions, dev, stream,
                           part_bytes + 2 * list_bytes + count_bytes + (size_t)units * sizeof(int), &ws))
        return rc;
    char* p = (char*)ws;
    a.part_o = (float*)p;
    a.part_ml = (float2*)(p + n_part * D * sizeof(float));
    p += part_bytes;
    int32_t* keys = (int32_t*)p;
    uint32_t* words = (uint32_t*)(p + list_bytes);
    int* counts = (int*)(p + 2 * list_bytes);
    a.flags = (int*)(p + 2 * list_bytes + count_bytes);
    a.keys = keys;
    a.words = words;
    a.counts = counts;
    a.q = q;
    a.k = k;
    a.v = v;
    a.khs = khs;
    a.krs = krs;
    a.vhs = vhs;
    a.vrs = vrs;
    a.out = out;
    a.L = n_rows;
    a.G = G;
    a.hkv = n_kv_heads;
    a.NR = NR;
    a.cap = cap;
    a.groups = groups;
    a.scale2 = scale * kLog2e;
    *flags = a.flags;
    const size_t plan_lds = (size_t)(std::min(n_keys, kPlanSeg) + 3) / 4 * 16;
    if (int rc = ensure_dynamic_lds((const void*)dlsa_plan_kernel, (size_t)kPlanSeg * sizeof(uint32_t)))
        return rc;
    hipLaunchKernelGGL(dlsa_plan_kernel, dim3(groups), dim3(kPlanThreads), plan_lds, stream, lists,
                       lengths, n_rows, width, n_keys, NR, KT, max_union, cap, n_kv_heads, keys, words,
                       counts, a.flags);
    QW_HIP_CHECK(hipGetLastError());
    const int grid = a.n_main + (groups - q_main) * n_kv_heads * a.n_split;
    a.q_dtype = q_dtype;
    if (rows32)
        return kv_dtype == QW_DTYPE_F32   ? launch_rows32<QW_DTYPE_F32>(a, D, grid, stream)
               : kv_dtype == QW_DTYPE_F16 ? launch_rows32<QW_DTYPE_F16>(a, D, grid, stream)
                                          : launch_rows32<QW_DTYPE_BF16>(a, D, grid, stream);
    if (bf16)
        return D == 256   ? launch_rows<256, true>(a, grid, stream)
               : D == 128 ? launch_rows<128, true>(a, grid, stream)
                          : launch_rows<64, true>(a, grid, stream);
    return D == 256   ? launch_rows<256, false>(a, grid, stream)
           : D == 128 ? launch_rows<128, false>(a, grid, stream)
                      : launch_rows<64, false>(a, grid, stream);
}

}  // namespace qw
