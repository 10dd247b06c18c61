// kv_cache.hip - KV cache lifecycle, quantize-on-append, dequantize and
// snapshot kernels for gfx950.
//
// Reference behaviour followed (cr0sh/qw):
//   KVCache::new_with_mode / update / update_and_fetch / trim / nbytes /
//   snapshot tensors: crates/mlxcel-core/src/cache.rs:526, :922-1157,
//   :2251-2300, :2709-2834, :3063, :570-626.
//   Affine codec (MLX `quantize` / `dequantize`, group 64):
//   crates/mlxcel-core/cpp/mlx_cxx_bridge.cpp:2991-3040, :6347-6393, at the
//   seam crates/mlxcel-core/src/cache/batch_quant.rs:109-158.
#include <string.h>

#include <algorithm>
#include <climits>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <type_traits>

#include "kv_cache.hpp"
#include "append.hpp"
#include "quant.hpp"
#include "rope.hpp"

namespace qw {

static thread_local std::string g_last_error;
void set_error(const std::string& msg) { g_last_error = msg; }
const char* last_error() { return g_last_error.c_str(); }

int GrowBuffer::get(size_t need, hipStream_t stream, void** out) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    QW_HIP_CHECK(hipStreamIsCapturing(stream, &cs));
    const bool capturing = cs != hipStreamCaptureStatusNone;
    if (need > bytes) {
        // HIP refuses allocation inside a global-mode capture, and the refused
        // call would invalidate the caller's capture: refuse here instead.
        QW_REQUIRE(!capturing, QW_ERR_STATE,
                   "split-K workspace: too small for this call and the stream is being captured; "
                   "run one call of this shape on this stream before capturing");
        if (ptr) {
            if (captured) {
                retired.push_back(ptr);  // a graph may still read it
            } else {
                if (stream_owned)
                    QW_HIP_CHECK(hipStreamSynchronize(stream));
                else
                    QW_HIP_CHECK(hipDeviceSynchronize());
                (void)hipFree(ptr);
            }
            ptr = nullptr;
            bytes = 0;
            captured = false;
        }
        const size_t nb = std::max(need + need / 4, (size_t)1 << 20);
        if (hipMalloc(&ptr, nb) != hipSuccess) {
            (void)hipGetLastError();
            ptr = nullptr;
            set_error("split-K workspace: hipMalloc failed");
            return QW_ERR_OUT_OF_MEMORY;
        }
        bytes = nb;
    }
    if (capturing) captured = true;
    *out = ptr;
    return QW_OK;
}

void GrowBuffer::release() {
    if (ptr) (void)hipFree(ptr);
    for (void* p : retired) (void)hipFree(p);
    retired.clear();
    ptr = nullptr;
    bytes = 0;
    captured = false;
}

// (nodes stay where they are: the map's lock covers the lookup alone, a buffer is its
// stream's, which the caller holds, and growth waits for that stream only)
static std::mutex g_ws_mu;
static std::map<std::tuple<int, hipStream_t, int>, GrowBuffer> g_ws;

int workspace(Workspace kind, int device, hipStream_t stream, size_t need, void** out) {
    GrowBuffer* b;
    {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        b = &g_ws[{device, stream, kind}];
    }
    b->stream_owned = true;
    return b->get(need, stream, out);
}

int release_workspaces(hipStream_t stream) {
    int dev = 0;
    QW_HIP_CHECK(hipGetDevice(&dev));
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    QW_HIP_CHECK(hipStreamIsCapturing(stream, &cs));
    QW_REQUIRE(cs == hipStreamCaptureStatusNone, QW_ERR_STATE,
               "release_workspaces: the stream is being captured");
    QW_HIP_CHECK(hipStreamSynchronize(stream));
    std::vector<GrowBuffer> freed;
    {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        for (int kind = 0; kind < kWorkspaces; kind++) {
            auto it = g_ws.find({dev, stream, kind});
            if (it == g_ws.end() || it->second.captured || !it->second.retired.empty()) continue;
            freed.push_back(it->second);
            g_ws.erase(it);
        }
    }
    for (GrowBuffer& b : freed) b.release();
    return QW_OK;
}

static std::mutex& stream_mutex(const void* stream) {
    static std::mutex mu[64];
    return mu[((uint64_t)(uintptr_t)stream * 0x9E3779B97F4A7C15ull) >> 58];
}
StreamLock::StreamLock(const void* stream) : lock(stream_mutex(stream)) {}

// Dynamic-LDS limits already raised, per (kernel, device). The attribute is
// a property of the kernel on the current device, so it is recorded per
// device, and the mutex keeps two host threads from interleaving a check and
// a set (which could leave the limit below what the record says).
static std::mutex g_lds_mu;
static std::map<std::pair<const void*, int>, size_t> g_lds_set;

int ensure_dynamic_lds(const void* kernel, size_t bytes) {
    if (bytes <= 65536) return QW_OK;  // the default limit
    int dev = 0;
    QW_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_lds_mu);
    size_t& cur = g_lds_set[{kernel, dev}];
    if (bytes <= cur) return QW_OK;
    QW_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    cur = bytes;
    return QW_OK;
}

// --------------------------------------------------------------- sizes

size_t KVCache::k_data_bytes(int c) const { return (size_t)hkv * c * D * bits / 8; }
size_t KVCache::k_param_bytes(int c) const {
    if (turbo4()) return (size_t)hkv * c * 4;
    return affine() ? (size_t)hkv * c * (D / kGroup) * 4 : 0;
}
size_t KVCache::v_data_bytes(int c) const { return (size_t)hkv * c * D * bits / 8; }
size_t KVCache::v_param_bytes(int c) const {
    if (turbo4()) return (size_t)hkv * (c / 8) * 32;
    return affine() ? (size_t)hkv * (c / 8) * (D / kGroup) * 32 : 0;
}

int64_t KVCache::nbytes() const {
    return (int64_t)(k_data_bytes(cap) + k_param_bytes(cap) + v_data_bytes(cap) +
                     v_param_bytes(cap));
}

static int round_cap(int capacity) {
    // The reference grows its buffers in steps of 256 tokens (cache.rs `step`).
    const int step = 256;
    return std::max(step, (capacity + step - 1) / step * step);
}

static int alloc_zero(void** p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0) return QW_OK;
    if (hipMalloc(p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        set_error("hipMalloc of " + std::to_string(bytes) + " bytes failed");
        return QW_ERR_OUT_OF_MEMORY;
    }
    // Zeroed so that rows past `offset` dequantize to finite zeros: masked keys
    // still pass through the P.V MFMA with weight 0.
    QW_HIP_CHECK(hipMemset(*p, 0, bytes));
    return QW_OK;
}

int KVCache::init(int mode_, int group_size, int n_kv_heads, int head_dim, int capacity,
                  int device_) {
    QW_REQUIRE(mode_ == QW_KV_FP16 || mode_ == QW_KV_AFFINE8 || mode_ == QW_KV_AFFINE4 ||
                   mode_ == QW_KV_INT8 || mode_ == QW_KV_TURBO4,
               QW_ERR_INVALID_ARGUMENT, "qw_kv_create: unknown mode");
    QW_REQUIRE(n_kv_heads > 0 && capacity >= 0 && head_dim > 0, QW_ERR_INVALID_ARGUMENT,
               "qw_kv_create: n_kv_heads, head_dim must be > 0 and capacity >= 0");
    if (mode_ == QW_KV_AFFINE8 || mode_ == QW_KV_AFFINE4) {
        QW_REQUIRE(group_size == kGroup, QW_ERR_UNSUPPORTED,
                   "qw_kv_create: affine modes use group_size 64");
        QW_REQUIRE(head_dim == 256 || head_dim == 128, QW_ERR_UNSUPPORTED,
                   "qw_kv_create: affine modes support head_dim 128 or 256");
    } else {
        // fp16, the per-token Int8 mode and Turbo4 have no group; group_size
        // is ignored
        QW_REQUIRE(head_dim == 256 || head_dim == 128, QW_ERR_UNSUPPORTED,
                   "qw_kv_create: fp16, int8 and turbo4 modes support head_dim 128 or 256");
    }
    mode = mode_;
    bits = (mode_ == QW_KV_AFFINE4 || mode_ == QW_KV_TURBO4) ? 4 : (mode_ == QW_KV_FP16 ? 16 : 8);
    D = head_dim;
    hkv = n_kv_heads;
    device = device_;
    offset = 0;
    cap = 0;
    DeviceGuard dg(device);
    QW_REQUIRE(dg.ok, QW_ERR_HIP, "qw_kv_create: hipSetDevice failed");
    if (hipMalloc(&fast_flag, 256) != hipSuccess) {
        (void)hipGetLastError();
        fast_flag = nullptr;
        set_error("qw_kv_create: hipMalloc failed");
        return QW_ERR_OUT_OF_MEMORY;
    }
    // Int8 codes always take the separately rounded dequant (offset 1152).
    const int fast0 = int8() ? 0 : 1;
    QW_HIP_CHECK(hipMemcpy(fast_flag, &fast0, sizeof(int), hipMemcpyHostToDevice));
    if (turbo4()) {
        int rc = turbo4_setup();
        if (rc) return rc;
    }
    return reserve(capacity, nullptr);
}

int KVCache::release() {
    DeviceGuard dg(device);
    (void)hipDeviceSynchronize();
    void* ptrs[6] = {k_data, (void*)k_params, v_data, (void*)v_params, (void*)fast_flag,
                     (void*)t4_tables};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    ws.release();
    fetch_ws.release();
    ws_ptr = nullptr;
    fast_flag = nullptr;
    t4_tables = nullptr;
    k_data = v_data = nullptr;
    k_params = v_params = nullptr;
    cap = offset = 0;
    return QW_OK;
}

int KVCache::reserve(int capacity, hipStream_t stream) {
    const int nc = round_cap(capacity);
    if (nc <= cap) return QW_OK;
    DeviceGuard dg(device);
    void *nk = nullptr, *nkp = nullptr, *nv = nullptr, *nvp = nullptr;
    int rc;
    if ((rc = alloc_zero(&nk, k_data_bytes(nc))) || (rc = alloc_zero(&nkp, k_param_bytes(nc))) ||
        (rc = alloc_zero(&nv, v_data_bytes(nc))) || (rc = alloc_zero(&nvp, v_param_bytes(nc)))) {
        void* ps[4] = {nk, nkp, nv, nvp};
        for (void* p : ps)
            if (p) (void)hipFree(p);
        return rc;
    }
    if (cap > 0) {
        // Per head, the first `cap` rows (K, K params) or cap/8 blocks (V, V
        // params) move to the head's start in the new buffers.
        // (Turbo4: row-major packed V, cap/8 blocks of 8 rows are the same
        // bytes; one 4-byte side record a row.)
        const size_t kr = (size_t)D * bits / 8;
        const size_t kpr = turbo4() ? 4 : (affine() ? (size_t)(D / kGroup) * 4 : 0);
        const size_t vb = (size_t)D * bits;
        const size_t vpb = turbo4() ? 32 : (affine() ? (size_t)(D / kGroup) * 32 : 0);
        for (int h = 0; h < hkv; h++) {
            QW_HIP_CHECK(hipMemcpyAsync((char*)nk + h * (size_t)nc * kr,
                                        (char*)k_data + h * (size_t)cap * kr, cap * kr,
                                        hipMemcpyDeviceToDevice, stream));
            QW_HIP_CHECK(hipMemcpyAsync((char*)nv + h * (size_t)(nc / 8) * vb,
                                        (char*)v_data + h * (size_t)(cap / 8) * vb,
                                        (cap / 8) * vb, hipMemcpyDeviceToDevice, stream));
            if (kpr) {
                QW_HIP_CHECK(hipMemcpyAsync((char*)nkp + h * (size_t)nc * kpr,
                                            (char*)k_params + h * (size_t)cap * kpr, cap * kpr,
                                            hipMemcpyDeviceToDevice, stream));
                QW_HIP_CHECK(hipMemcpyAsync((char*)nvp + h * (size_t)(nc / 8) * vpb,
                                            (char*)v_params + h * (size_t)(cap / 8) * vpb,
                                            (cap / 8) * vpb, hipMemcpyDeviceToDevice, stream));
            }
        }
        QW_HIP_CHECK(hipStreamSynchronize(stream));
        void* old[4] = {k_data, (void*)k_params, v_data, (void*)v_params};
        for (void* p : old)
            if (p) (void)hipFree(p);
    }
    k_data = nk;
    k_params = (uint32_t*)nkp;
    v_data = nv;
    v_params = (uint32_t*)nvp;
    cap = nc;
    return QW_OK;
}

int KVCache::ensure_workspace(size_t bytes, hipStream_t stream) {
    DeviceGuard dg(device);
    return ws.get(bytes, stream, &ws_ptr);
}

int KVCache::demote(int target_mode, hipStream_t stream, int* demoted) {
    // cache.rs:3591 demote_fp16_to_turbo4: a populated fp16 cache is re-stored
    // in the quantized mode by quantize-appending its rows [0, offset) to an
    // empty cache of that mode; anything else is left alone (returns 0).
    *demoted = 0;
    QW_REQUIRE(target_mode == QW_KV_AFFINE4 || target_mode == QW_KV_AFFINE8 ||
                   target_mode == QW_KV_TURBO4,
               QW_ERR_INVALID_ARGUMENT, "demote: target mode must be an affine mode or turbo4");
    if (mode != QW_KV_FP16 || offset <= 0) return QW_OK;
    DeviceGuard dg(device);
    QW_REQUIRE(dg.ok, QW_ERR_HIP, "demote: hipSetDevice failed");
    const int n = offset;
    const size_t bytes = (size_t)hkv * n * D * sizeof(f16);
    void *tk = nullptr, *tv = nullptr;
    if (hipMalloc(&tk, bytes) != hipSuccess || hipMalloc(&tv, bytes) != hipSuccess) {
        (void)hipGetLastError();
        if (tk) (void)hipFree(tk);
        set_error("demote: hipMalloc of the fp16 staging rows failed");
        return QW_ERR_OUT_OF_MEMORY;
    }
    int rc = dequantize(0, n, tk, tv, stream);  // the fp16 rows, [hkv][n][D]
    if (rc == QW_OK) rc = hipStreamSynchronize(stream) == hipSuccess ? QW_OK : QW_ERR_HIP;
    if (rc) {
        (void)hipFree(tk);
        (void)hipFree(tv);
        return rc;
    }
    void* old[4] = {k_data, (void*)k_params, v_data, (void*)v_params};
    const int old_cap = cap;
    k_data = v_data = nullptr;
    k_params = v_params = nullptr;
    cap = 0;
    offset = 0;
    mode = target_mode;
    bits = target_mode == QW_KV_AFFINE8 ? 8 : 4;
    rc = turbo4() ? turbo4_setup() : QW_OK;
    if (rc == QW_OK) rc = reserve(old_cap, stream);
    if (rc == QW_OK) rc = update(tk, tv, n, stream);
    if (rc == QW_OK) rc = hipStreamSynchronize(stream) == hipSuccess ? QW_OK : QW_ERR_HIP;
    (void)hipFree(tk);
    (void)hipFree(tv);
    if (rc) return rc;  // the cache is left empty in the new mode
    for (void* p : old)
        if (p) (void)hipFree(p);
    *demoted = 1;
    return QW_OK;
}

int KVCache::trim(int n) {
    // cache.rs:2251: clamp to the cached length; buffers keep their rows, the
    // next append overwrites them.
    const int m = std::min(n, offset);
    if (m <= 0) return 0;
    offset -= m;
    return m;
}

// Quantize-on-append: one workgroup (4 waves) per (8-token V block touched by
// the append, KV head).
template <int D>
__global__ __launch_bounds__(256) void append_affine_kernel(
    RowSrc rs, int n_tokens, int t_old,
    int bits, int int8, int cap, uint32_t* __restrict__ k_codes, uint32_t* __restrict__ k_params,
    uint32_t* __restrict__ v_codes, f16* __restrict__ v_params, int* __restrict__ fast_flag) {
    __shared__ AppendScratch<D> sc;
    append_block<D>(rs, n_tokens, t_old, bits, int8 != 0, cap, k_codes, k_params, v_codes, v_params,
                    fast_flag, t_old / 8 + blockIdx.x, blockIdx.y, threadIdx.x, blockDim.x, sc);
}

// The same for many tokens of the affine modes: a thread takes 8 dims of the 8 tokens
// of one V block, of K or of V (16-byte loads, all issued first), and forms their
// codes in registers: a group is 8 lanes, its extremes three lane moves a token; lane
// i of them forms token i's scale and bias for all (the divisions once a group, where
// every lane of the row-wise form divides) and hands them round; the words of a K row
// and of the V block's dims are assembled in place and stored whole (V in 16-byte
// pieces). A workgroup that meets a value that is not finite leaves its blocks to the
// row-wise form (append_block; the other plane's workgroup stores the same bytes), so
// such rows are stored as before. VALU-bound, two waves a SIMD (about 200
// registers): 65536 tokens of 4 heads, D = 256, 4-bit 203 us row-wise -> 125 us, 2048
// tokens 11.4 -> 8.9 us; 8 heads, D = 128, 8-bit 313 -> 131 us. (Int8's codes have no
// division to share: 363 -> 376 us at 131072 tokens, so it stays row-wise.)
template <int D, int BITS>
__global__ __launch_bounds__(256) void append_affine_blocks_kernel(
    RowSrc rs, int n_tokens, int t_old, int cap, uint32_t* __restrict__ k_codes,
    uint32_t* __restrict__ k_params, uint32_t* __restrict__ v_codes, f16* __restrict__ v_params,
    int* __restrict__ fast_flag) {
    constexpr int OCT = D / 8, NG = D / kGroup, BPW = 256 / OCT;  // blocks a workgroup
    constexpr int E = 16 / BITS, NV = BITS / 2;                   // dims a piece of V, pieces
    __shared__ AppendScratch<D> sc;
    const int tid = threadIdx.x, h = blockIdx.y, lane = tid & 63, l8 = lane & 7;
    const bool is_v = blockIdx.z != 0;
    const int b_first = t_old / 8, b_last = (t_old + n_tokens - 1) / 8;
    const int blk = b_first + blockIdx.x * BPW + tid / OCT, d0 = tid % OCT * 8, grp = d0 / kGroup;
    const int r0 = 8 * blk - t_old;  // the source row of the block's first key
    const bool live = blk <= b_last;
    half8 x[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int r = min(max(r0 + i, 0), n_tokens - 1);
        const int64_t src = (int64_t)r * rs.row_stride + (int64_t)h * rs.head_stride + d0;
        x[i] = *(const half8*)((is_v ? rs.v : rs.k) + src);
    }
    const int64_t gblk = (int64_t)h * (cap / 8) + (live ? blk : b_last);
    u32x4* const vw = (u32x4*)(v_codes + gblk * (D * BITS / 4));
    u32x4 w[NV];  // the 8 dims' words of the V block, in pieces; earlier tokens' codes stay
#pragma unroll
    for (int j = 0; j < NV; j++) {
        w[j] = u32x4{0, 0, 0, 0};
        if (is_v && live && r0 < 0) w[j] = vw[v_phys_dim(d0 + E * j, D, BITS) / E];
    }
    bool odd = false;
    float my_mn = 0.0f, my_mx = 0.0f;  // token l8's extremes in this lane's group
#pragma unroll
    for (int i = 0; i < 8; i++) {
        float mx = (float)x[i][0], mn = mx;
        odd |= !(fabsf(mx) < INFINITY);
#pragma unroll
        for (int e = 1; e < 8; e++) {
            const float f = (float)x[i][e];
            odd |= !(fabsf(f) < INFINITY);
            mx = fmaxf(mx, f);
            mn = fminf(mn, f);
        }
        mx = fmaxf(mx, lane_xor<1>(mx, lane));
        mn = fminf(mn, lane_xor<1>(mn, lane));
        mx = fmaxf(mx, lane_xor<2>(mx, lane));
        mn = fminf(mn, lane_xor<2>(mn, lane));
        mx = fmaxf(mx, lane_xor<4>(mx, lane));
        mn = fminf(mn, lane_xor<4>(mn, lane));
        if (i == l8) {
            my_mx = mx;
            my_mn = mn;
        }
    }
    if (__syncthreads_or(odd)) {
        for (int b = 0; b < BPW; b++) {
            const int bb = b_first + blockIdx.x * BPW + b;
            if (bb > b_last) break;
            append_block<D>(rs, n_tokens, t_old, BITS, false, cap, k_codes, k_params, v_codes, v_params,
                            fast_flag, bb, h, tid, 256, sc);
            __syncthreads();
        }
        return;
    }
    // the halves are converted again below: their floats are not held over the scan
#pragma unroll
    for (int i = 0; i < 8; i++) asm volatile("" : "+v"(x[i]));
    const AffineGroup q = affine_group(my_mn, my_mx, BITS);
    const float inv = 1.0f / q.scale;
    if (live && r0 + l8 >= 0 && r0 + l8 < n_tokens) {
        half2v sb;
        sb.x = (f16)q.scale;
        sb.y = (f16)q.bias;
        check_fast_scale(sb.x, BITS, fast_flag);
        if (is_v) {
            f16* vp = v_params + (gblk * NG + grp) * 16;
            vp[l8] = sb.x;
            vp[8 + l8] = sb.y;
        } else {
            k_params[(gblk * 8 + l8) * NG + k_param_slot(grp, NG)] = __builtin_bit_cast(uint32_t, sb);
        }
    }
    const int base = lane & ~7;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const AffineGroup qi{__shfl(q.scale, base + i), __shfl(q.bias, base + i)};
        const float ii = __shfl(inv, base + i);
        const bool ok = live && r0 + i >= 0 && r0 + i < n_tokens;
        uint32_t c[8];
#pragma unroll
        for (int e = 0; e < 8; e++) c[e] = (uint32_t)affine_code_inv((float)x[i][e], qi, ii, BITS);
        if (!ok) continue;
        if (!is_v) {
            uint32_t* row = k_codes + ((gblk * 8 + i) * D + d0) * BITS / 32;
            if constexpr (BITS == 4) {
                uint32_t word = 0;
#pragma unroll
                for (int e = 0; e < 8; e++) word |= c[e] << (4 * e);
                *row = word;
            } else {
                *(u32x2*)row = u32x2{c[0] | (c[1] << 8) | (c[2] << 16) | (c[3] << 24),
                                     c[4] | (c[5] << 8) | (c[6] << 16) | (c[7] << 24)};
            }
        } else {
            const int sh = BITS == 4 ? 4 * v4_nibble_pos(i) : 8 * (i & 3);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int at = BITS == 4 ? e & 3 : 2 * (e & 1) + i / 4;
                const uint32_t m = ((1u << BITS) - 1u) << sh;
                w[e / E][at] = (w[e / E][at] & ~m) | (c[e] << sh);
            }
        }
    }
    if (is_v && live) {
#pragma unroll
        for (int j = 0; j < NV; j++) vw[v_phys_dim(d0 + E * j, D, BITS) / E] = w[j];
    }
}

// fp16 mode append: K rows copied, V transposed into 8-key blocks. A thread takes
// 8 dims of one block's 8 tokens: 16-byte loads of both (all issued first), K rows
// stored as they are, a dim's 8 keys of V as one 16-byte piece where the append
// fills the block (single elements where it does not). HBM-bound; 131072 rows of 4
// heads, D = 256: 730 us an element a thread -> 198 us.
template <int D>
__global__ __launch_bounds__(256) void append_fp16_kernel(RowSrc rs, int n_tokens, int t_old,
                                                          int cap, f16* __restrict__ k_data,
                                                          f16* __restrict__ v_data) {
    constexpr int OCT = D / 8;
    const int h = blockIdx.y, unit = blockIdx.x * 256 + threadIdx.x;
    const int blk = t_old / 8 + unit / OCT, d0 = unit % OCT * 8;
    const int r0 = 8 * blk - t_old;  // the source row of the block's first key
    if (r0 >= n_tokens) return;
    // (rows and pieces off 16 bytes: the caller's pointers and strides decide)
    const bool wide = (((uintptr_t)rs.k | (uintptr_t)rs.v) % 16 == 0) && rs.row_stride % 8 == 0 &&
                      rs.head_stride % 8 == 0;
    half8 kr[8], vr[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int r = min(max(r0 + i, 0), n_tokens - 1);
        const int64_t src = (int64_t)r * rs.row_stride + (int64_t)h * rs.head_stride + d0;
        if (wide) {
            kr[i] = *(const half8*)(rs.k + src);
            vr[i] = *(const half8*)(rs.v + src);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                kr[i][e] = rs.k[src + e];
                vr[i][e] = rs.v[src + e];
            }
        }
    }
    const int64_t gblk = (int64_t)h * (cap / 8) + blk;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int r = r0 + i;
        if (r < 0 || r >= n_tokens) continue;
        *(half8*)(k_data + (gblk * 8 + i) * D + d0) = kr[i];
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
        f16* p = v_data + (gblk * D + v_phys_dim(d0 + e, D, 16)) * 8;
        if (r0 >= 0 && r0 + 8 <= n_tokens) {
            half8 y;
#pragma unroll
            for (int i = 0; i < 8; i++) y[i] = vr[i][e];
            *(half8*)p = y;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (r0 + i >= 0 && r0 + i < n_tokens) p[i] = vr[i][e];
        }
    }
}

// The same with an element a thread: K rotated on the load (the library's sine and
// cosine are most of the work), and shorter appends, below kBlockCopy.
template <int D>
__global__ __launch_bounds__(256) void append_fp16_elem_kernel(RowSrc rs, int n_tokens, int t_old,
                                                          int cap, f16* __restrict__ k_data,
                                                          f16* __restrict__ v_data) {
    const int h = blockIdx.y;
    const int64_t n = (int64_t)n_tokens * D;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(i / D), d = (int)(i % D);
        const int t = r + t_old;
        const int64_t src = (int64_t)r * rs.row_stride + (int64_t)h * rs.head_stride;
        const f16 kv = (f16)rope_elem(rs.k + src, d, rs.rope_dims, rs.traditional, rs.log2_base,
                                      rs.scale, rs.position0 + r);
        const f16 vv = rs.v[src + d];
        k_data[((int64_t)h * cap + t) * D + d] = kv;
        v_data[(((int64_t)h * (cap / 8) + t / 8) * D + v_phys_dim(d, D, 16)) * 8 + (t & 7)] = vv;
    }
}

int KVCache::update(const void* k_new, const void* v_new, int n_tokens, hipStream_t stream) {
    QW_REQUIRE(n_tokens >= 0, QW_ERR_INVALID_ARGUMENT, "update: n_tokens must be >= 0");
    if (n_tokens == 0) return QW_OK;
    QW_REQUIRE(k_new && v_new, QW_ERR_INVALID_ARGUMENT, "update: null K/V pointer");
    RowSrc rs{};
    rs.k = (const f16*)k_new;
    rs.v = (const f16*)v_new;
    rs.row_stride = D;
    rs.head_stride = (int64_t)n_tokens * D;
    return update_rows(rs, n_tokens, stream);
}

// Halves of K from which an affine append takes the block-wise form (below it its few long
// chains cost more than the row-wise form's divisions): 4-bit, D = 256, 4 heads, row-wise
// against it, 700 tokens 8.0 / 8.4 us, 1024 8.2 / 8.5, 1500 9.5 / 8.7, 4096 18.0 / 15.0;
// 2 heads, 2048 tokens 8.5 / 8.6, 4096 12.2 / 10.0; 16 heads, 512 tokens 12.0 / 9.8.
constexpr int64_t kBlockAppend = 5 << 18;
// And an fp16 append, which starts whole blocks (offset % 8 == 0) / which does not (single
// halves of V): fewer threads of longer chains cost 1 us / 2.5 us more until the element
// form's 2-byte stores cost that. An element a thread against it, 4 heads, D = 256: 8
// tokens 3.2 / 3.9 us (off a block 3.2 / 5.8), 256 4.3 / 4.3 (4.3 / 5.7), 512 5.5 / 4.4 (5.5 /
// 5.8), 1024 7.5 / 4.7 (7.6 / 6.0); 8 heads, D = 128, 512 tokens 4.6 / 4.4 (4.9 / 5.8); 16
// heads, D = 256, 128 tokens 5.5 / 4.4 (5.5 / 5.9); the same at 1 and 2 heads by bytes.
constexpr int64_t kBlockCopy = 3 << 17, kBlockCopyOff = 3 << 18;

int KVCache::update_rows(const RowSrc& rs, int n_tokens, hipStream_t stream) {
    if (n_tokens == 0) return QW_OK;
    DeviceGuard dg(device);
    QW_REQUIRE(dg.ok, QW_ERR_HIP, "update: hipSetDevice failed");
    const int need = offset + n_tokens;
    if (need > cap) {
        // Geometric growth keeps appends amortized O(1) per token.
        int rc = reserve(std::max(need, cap + cap / 2), stream);
        if (rc) return rc;
    }
    if (turbo4()) {
        int rc = turbo4_update(rs, n_tokens, stream);
        if (rc) return rc;
    } else if (affine()) {
        const int nblk = (offset + n_tokens - 1) / 8 - offset / 8 + 1;
        dim3 grid(nblk, hkv);
        // many rows as they are, their pieces on 16 bytes: the block-wise form
        if ((int64_t)n_tokens * hkv * D >= kBlockAppend && !int8() && rs.rope_dims == 0 &&
            (((uintptr_t)rs.k | (uintptr_t)rs.v) % 16 == 0) && rs.row_stride % 8 == 0 &&
            rs.head_stride % 8 == 0) {
            const int bpw = 256 / (D / 8);
            grid = dim3((nblk + bpw - 1) / bpw, hkv, 2);
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, rs, n_tokens, offset, cap,
                                   (uint32_t*)k_data, k_params, (uint32_t*)v_data, (f16*)v_params,
                                   fast_flag);
            };
            if (D == 256)
                bits == 8 ? launch(append_affine_blocks_kernel<256, 8>)
                          : launch(append_affine_blocks_kernel<256, 4>);
            else
                bits == 8 ? launch(append_affine_blocks_kernel<128, 8>)
                          : launch(append_affine_blocks_kernel<128, 4>);
        } else if (D == 256)
            hipLaunchKernelGGL(append_affine_kernel<256>, grid, dim3(256), 0, stream,
                               rs, n_tokens, offset, bits,
                               int8() ? 1 : 0, cap, (uint32_t*)k_data, k_params,
                               (uint32_t*)v_data, (f16*)v_params, fast_flag);
        else
            hipLaunchKernelGGL(append_affine_kernel<128>, grid, dim3(256), 0, stream,
                               rs, n_tokens, offset, bits,
                               int8() ? 1 : 0, cap, (uint32_t*)k_data, k_params,
                               (uint32_t*)v_data, (f16*)v_params, fast_flag);
    } else {
        const int nblk = (offset + n_tokens - 1) / 8 - offset / 8 + 1;
        const bool elem = rs.rope_dims > 0 ||
                          (int64_t)n_tokens * hkv * D < (offset % 8 ? kBlockCopyOff : kBlockCopy);
        const int64_t threads = elem ? (int64_t)n_tokens * D : (int64_t)nblk * (D / 8);
        const dim3 grid((unsigned)std::min<int64_t>((threads + 255) / 256, elem ? 1024 : INT_MAX), hkv);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, rs, n_tokens, offset, cap,
                               (f16*)k_data, (f16*)v_data);
        };
        if (D == 256)
            elem ? launch(append_fp16_elem_kernel<256>) : launch(append_fp16_kernel<256>);
        else
            elem ? launch(append_fp16_elem_kernel<128>) : launch(append_fp16_kernel<128>);
    }
    QW_HIP_CHECK(hipGetLastError());
    offset += n_tokens;
    return QW_OK;
}

// ------------------------------------------------------------ dequantize
//
// MLX's composite dequantize: out = f16(f16(code * scale) + bias). code *
// scale is exact in fp32 (<= 8 x 11 significant bits), so the first cast is
// the fp16 product; the sum is formed in fp32 and cast once more, which is
// how MLX's CPU float16 type evaluates `a + b`.

// `off` is 128 for Int8 codes stored biased by 128 (bias 0: the result is
// f16(code * scale), the reference's Int8 dequantize, cache.rs:313-316).
__device__ inline f16 mlx_dequant(uint32_t c, int off, f16 s, f16 b) {
    const f16 prod = (f16)((float)((int)c - off) * (float)s);
    return (f16)((float)prod + (float)b);
}

// A thread takes 8 dims of the 8 keys of one V block: V's codes (fp16: values) as
// 16-byte pieces that hold all 8 keys of a dim or two, K's as one word or two (16
// bytes) a key, every load issued before the first is used; then a 16-byte store a
// key and plane, 64 lanes covering whole rows. HBM-bound: 8192 rows of 4 heads, D =
// 256, 4-bit (9.4 MB in, 33.6 out) in 8.8 us; one key a thread, each element's code
// gathered for itself, took 26.4 us. Short windows leave the chip to few such threads
// (64 rows 4.6 us): there a thread of KPT = 1 forms one key of the eight (3.3 us; 512 rows
// 4.9 / 4.9, 2048 rows 5.7 in blocks).
template <int BITS, int D, int KPT>
__global__ __launch_bounds__(256) void fetch_kernel(const void* __restrict__ k_data,
                                                    const uint32_t* __restrict__ k_params,
                                                    const void* __restrict__ v_data,
                                                    const f16* __restrict__ v_params, int code_off,
                                                    int cap, int start, int n,
                                                    f16* __restrict__ k_out,
                                                    f16* __restrict__ v_out) {
    constexpr int OCT = D / 8, NG = D / kGroup;
    constexpr int NV = BITS / 2;       // 16-byte pieces of V
    constexpr int E = 16 / BITS;       // dims a piece
    constexpr int KW = BITS / 4;       // words of 8 dims of a K row
    const int h = blockIdx.y, unit = blockIdx.x * 256 + threadIdx.x;
    const int d0 = unit % OCT * 8, g = d0 / kGroup, first = start / 8 * 8 + unit / OCT * KPT;
    const int blk = first / 8, k0 = KPT == 8 ? 0 : first % 8;  // (keys k0 .. k0 + KPT - 1 of the block)
    if (first >= start + n) return;
    const int64_t gblk = (int64_t)h * (cap / 8) + blk;
    u32x4 vc[NV];
#pragma unroll
    for (int j = 0; j < NV; j++)
        vc[j] = ((const u32x4*)v_data)[(gblk * D + v_phys_dim(d0 + E * j, D, BITS)) / E];
    u32x4 vs = {}, vb = {};
    if constexpr (BITS != 16) {
        const u32x4* vp = (const u32x4*)(v_params + (gblk * NG + g) * 16);
        vs = vp[0];
        vb = vp[1];
    }
    uint32_t kc[KPT][KW], ksb[KPT] = {};
#pragma unroll
    for (int k = 0; k < KPT; k++) {
        const int64_t row = gblk * 8 + k0 + k;  // (rows of a block exist up to cap)
        const uint32_t* p = (const uint32_t*)k_data + (row * D + d0) * BITS / 32;
#pragma unroll
        for (int w = 0; w < KW; w++) kc[k][w] = p[w];
        if constexpr (BITS != 16) ksb[k] = k_params[row * NG + k_param_slot(g, NG)];
    }
#pragma unroll
    for (int i = 0; i < KPT; i++) {
        const int k = k0 + i, r = 8 * blk + k - start;
        if (r < 0 || r >= n) continue;
        half8 ko, vo;
        const half2v sb = h2(ksb[i]);
        const f16 s = h2(vs[k / 2])[k & 1], b = h2(vb[k / 2])[k & 1];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            // piece e / E holds dims in turn, each 32 / 64 / 128 bits of 8 keys
            const u32x4 w = vc[e / E];
            if constexpr (BITS == 16) {
                ko[e] = h2(kc[i][e / 2])[e & 1];
                vo[e] = h2(w[k / 2])[k & 1];
            } else if constexpr (BITS == 8) {
                ko[e] = mlx_dequant((kc[i][e / 4] >> (8 * (e & 3))) & 0xFFu, code_off, sb.x, sb.y);
                vo[e] = mlx_dequant((w[2 * (e & 1) + k / 4] >> (8 * (k & 3))) & 0xFFu, code_off, s, b);
            } else {
                ko[e] = mlx_dequant((kc[i][0] >> (4 * e)) & 0xFu, code_off, sb.x, sb.y);
                vo[e] = mlx_dequant((w[e & 3] >> (4 * v4_nibble_pos(k))) & 0xFu, code_off, s, b);
            }
        }
        const int64_t o = ((int64_t)h * n + r) * D + d0;
        *(half8*)(k_out + o) = ko;
        *(half8*)(v_out + o) = vo;
    }
}

constexpr int64_t kShortFetch = 1 << 19;  // halves of K

// fp16 mode into outputs off 16-byte alignment: element by element.
__global__ __launch_bounds__(256) void fetch_fp16_kernel(const f16* __restrict__ k_data,
                                                         const f16* __restrict__ v_data, int D,
                                                         int cap, int hkv, int start, int n,
                                                         f16* __restrict__ k_out,
                                                         f16* __restrict__ v_out) {
    const int64_t total = (int64_t)hkv * n * D;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int h = (int)(i / ((int64_t)n * D));
        const int r = (int)((i / D) % n);
        const int d = (int)(i % D);
        const int t = start + r;
        k_out[i] = k_data[((int64_t)h * cap + t) * D + d];
        v_out[i] =
            v_data[(((int64_t)h * (cap / 8) + t / 8) * D + v_phys_dim(d, D, 16)) * 8 + (t & 7)];
    }
}

int KVCache::dequantize(int start, int n, void* k_out, void* v_out, hipStream_t stream) const {
    QW_REQUIRE(start >= 0 && n >= 0 && start + n <= offset, QW_ERR_INVALID_ARGUMENT,
               "dequantize: window [start, start+n) outside the cached rows");
    if (n == 0) return QW_OK;
    QW_REQUIRE(k_out && v_out, QW_ERR_INVALID_ARGUMENT, "dequantize: null output");
    DeviceGuard dg(device);
    if (turbo4()) return turbo4_dequantize(start, n, k_out, v_out, stream);
    if (!affine() && (((uintptr_t)k_out | (uintptr_t)v_out) % 16) != 0) {
        const unsigned blocks = (unsigned)std::min<int64_t>(((int64_t)hkv * n * D + 255) / 256, 4096);
        hipLaunchKernelGGL(fetch_fp16_kernel, dim3(blocks), dim3(256), 0, stream,
                           (const f16*)k_data, (const f16*)v_data, D, cap, hkv, start, n,
                           (f16*)k_out, (f16*)v_out);
        QW_HIP_CHECK(hipGetLastError());
        return QW_OK;
    }
    const int nblk = (start + n - 1) / 8 - start / 8 + 1;
    auto run = [&](auto kpt) {
        constexpr int KPT = decltype(kpt)::value;
        const dim3 grid((unsigned)(((int64_t)nblk * (8 / KPT) * (D / 8) + 255) / 256), hkv);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, k_data, k_params, v_data,
                               (const f16*)v_params, int8() ? 128 : 0, cap, start, n, (f16*)k_out,
                               (f16*)v_out);
        };
        if (D == 256)
            bits == 4 ? launch(fetch_kernel<4, 256, KPT>)
                      : bits == 8 ? launch(fetch_kernel<8, 256, KPT>) : launch(fetch_kernel<16, 256, KPT>);
        else
            bits == 4 ? launch(fetch_kernel<4, 128, KPT>)
                      : bits == 8 ? launch(fetch_kernel<8, 128, KPT>) : launch(fetch_kernel<16, 128, KPT>);
    };
    if ((int64_t)n * hkv * D < kShortFetch)
        run(std::integral_constant<int, 1>{});
    else
        run(std::integral_constant<int, 8>{});
    QW_HIP_CHECK(hipGetLastError());
    return QW_OK;
}

int KVCache::update_and_fetch(const void* k_new, const void* v_new, int n_tokens, void* k_out,
                              void* v_out, hipStream_t stream) {
    int rc = update(k_new, v_new, n_tokens, stream);
    if (rc) return rc;
    return dequantize(0, offset, k_out, v_out, stream);
}

// ------------------------------------------------------- snapshot tensors
//
// Export/import in the reference's layout: per head, rows [0, offset) of
// MLX-packed codes and separate fp16 scale and bias planes (cache.rs:570-626
// exports packed tensors as they are, without requantizing).

// V blocks <-> rows, plus the K param split/merge. dir = 0: export.
// Int8 mode: codes leave and enter as signed bytes (stored + 128, i.e. XOR
// 0x80 per byte) and one scale per row (the first group's; every group holds
// it, with bias 0).
__global__ __launch_bounds__(256) void snapshot_affine_kernel(
    int dir, int bits, int int8, int D, int cap, int hkv, int n, int* __restrict__ fast_flag,
    uint32_t* __restrict__ k_params,
    uint32_t* __restrict__ v_codes, f16* __restrict__ v_params, f16* __restrict__ ks_out,
    f16* __restrict__ kb_out, uint32_t* __restrict__ vc_rows, f16* __restrict__ vs_rows,
    f16* __restrict__ vb_rows) {
    const int NG = D / kGroup;
    const int nw = D * bits / 32;
    const int epw = 32 / bits;
    const uint32_t m = (1u << bits) - 1u;
    const int64_t total = (int64_t)hkv * n * nw;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int h = (int)(i / ((int64_t)n * nw));
        const int t = (int)((i / nw) % n);
        const int w = (int)(i % nw);
        const int k = t & 7;
        uint32_t* vblk = v_codes + ((int64_t)h * (cap / 8) + t / 8) * (D * bits / 4);
        const int64_t row = (int64_t)h * n + t;
        if (dir == 0) {
            uint32_t word = 0;
            for (int e = 0; e < epw; e++) {
                const int p = v_phys_dim(w * epw + e, D, bits);
                const uint32_t c = bits == 4 ? (vblk[p] >> (4 * v4_nibble_pos(k))) & m
                                             : (vblk[2 * p + (k >> 2)] >> (8 * (k & 3))) & m;
                word |= c << (e * bits);
            }
            vc_rows[row * nw + w] = int8 ? word ^ 0x80808080u : word;
        }
        if (w < NG) {
            const int g = w;
            const int64_t kp = ((int64_t)h * cap + t) * NG + k_param_slot(g, NG);
            f16* vp = v_params + (((int64_t)h * (cap / 8) + t / 8) * NG + g) * 16;
            if (int8) {
                if (dir == 0) {
                    if (g == 0) {
                        ks_out[row] = __builtin_bit_cast(half2v, k_params[kp]).x;
                        vs_rows[row] = vp[k];
                    }
                } else {
                    half2v sb;
                    sb.x = ks_out[row];
                    sb.y = (f16)0.0f;
                    k_params[kp] = __builtin_bit_cast(uint32_t, sb);
                    vp[k] = vs_rows[row];
                    vp[8 + k] = (f16)0.0f;
                }
            } else if (dir == 0) {
                const half2v sb = __builtin_bit_cast(half2v, k_params[kp]);
                ks_out[row * NG + g] = sb.x;
                kb_out[row * NG + g] = sb.y;
                vs_rows[row * NG + g] = vp[k];
                vb_rows[row * NG + g] = vp[8 + k];
            } else {
                half2v sb;
                sb.x = ks_out[row * NG + g];
                sb.y = kb_out[row * NG + g];
                k_params[kp] = __builtin_bit_cast(uint32_t, sb);
                vp[k] = vs_rows[row * NG + g];
                vp[8 + k] = vb_rows[row * NG + g];
                check_fast_scale(sb.x, bits, fast_flag);
                check_fast_scale(vp[k], bits, fast_flag);
            }
        }
    }
}

__global__ void set_flag_kernel(int* flag, int v) { *flag = v; }

// Import of V codes: one thread per (head, block, dim) builds the block word(s).
__global__ __launch_bounds__(256) void import_v_codes_kernel(int bits, int int8, int D, int cap,
                                                             int hkv, int n,
                                                             const uint32_t* __restrict__ rows,
                                                             uint32_t* __restrict__ v_codes) {
    const int nblk = (n + 7) / 8;
    const int nw = D * bits / 32;
    const int epw = 32 / bits;
    const uint32_t m = (1u << bits) - 1u;
    const int64_t total = (int64_t)hkv * nblk * D;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int h = (int)(i / ((int64_t)nblk * D));
        const int b = (int)((i / D) % nblk);
        const int d = (int)(i % D);
        uint32_t w0 = 0, w1 = 0;
        for (int k = 0; k < 8; k++) {
            const int t = b * 8 + k;
            if (t >= n) break;
            const uint32_t c = (rows[((int64_t)h * n + t) * nw + d / epw] >> ((d % epw) * bits)) & m;
            if (bits == 4)
                w0 |= c << (4 * v4_nibble_pos(k));
            else if (k < 4)
                w0 |= c << (8 * k);
            else
                w1 |= c << (8 * (k - 4));
        }
        if (int8) {
            // Int8: signed bytes in, biased bytes stored (slots past n stay 128 = code 0)
            w0 ^= 0x80808080u;
            w1 ^= 0x80808080u;
        }
        uint32_t* vblk = v_codes + ((int64_t)h * (cap / 8) + b) * (D * bits / 4);
        const int p = v_phys_dim(d, D, bits);
        if (bits == 4) {
            vblk[p] = w0;
        } else {
            vblk[2 * p] = w0;
            vblk[2 * p + 1] = w1;
        }
    }
}

// XOR 0x80 into every byte of rows [0, n) of each head's row-major K codes
// ([hkv][stride][nw] words): signed <-> biased Int8 codes.
__global__ __launch_bounds__(256) void flip_code_sign_kernel(uint32_t* __restrict__ words, int hkv,
                                                             int n, int nw, int stride) {
    const int64_t total = (int64_t)hkv * n * nw;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int h = (int)(i / ((int64_t)n * nw));
        const int64_t r = i % ((int64_t)n * nw);
        words[(int64_t)h * stride * nw + r] ^= 0x80808080u;
    }
}

int KVCache::export_tensors(void* k_codes, void* k_scales, void* k_biases, void* v_codes,
                            void* v_scales, void* v_biases, hipStream_t stream) const {
    QW_REQUIRE(!turbo4(), QW_ERR_STATE, "export: a Turbo4 cache exports with qw_kv_export_turbo4");
    QW_REQUIRE(k_codes && v_codes, QW_ERR_INVALID_ARGUMENT, "export: null code pointers");
    QW_REQUIRE(!affine() || (k_scales && v_scales && (int8() || (k_biases && v_biases))),
               QW_ERR_INVALID_ARGUMENT, "export: null scale/bias pointers");
    if (offset == 0) return QW_OK;
    DeviceGuard dg(device);
    const int n = offset;
    if (!affine()) {
        // Same as a full fetch in fp16 mode.
        return dequantize(0, n, k_codes, v_codes, stream);
    }
    const size_t kr = (size_t)D * bits / 8;
    for (int h = 0; h < hkv; h++)
        QW_HIP_CHECK(hipMemcpyAsync((char*)k_codes + h * (size_t)n * kr,
                                    (const char*)k_data + h * (size_t)cap * kr, n * kr,
                                    hipMemcpyDeviceToDevice, stream));
    const int64_t work = (int64_t)hkv * n * (D * bits / 32);
    const unsigned nb = (unsigned)std::min<int64_t>((work + 255) / 256, 4096);
    if (int8()) {
        hipLaunchKernelGGL(flip_code_sign_kernel, dim3(nb), dim3(256), 0, stream,
                           (uint32_t*)k_codes, hkv, n, D / 4, n);
        QW_HIP_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL(snapshot_affine_kernel, dim3(nb), dim3(256), 0, stream, 0, bits,
                       int8() ? 1 : 0, D, cap, hkv, n, fast_flag, k_params, (uint32_t*)v_data,
                       (f16*)v_params, (f16*)k_scales, (f16*)k_biases, (uint32_t*)v_codes,
                       (f16*)v_scales, (f16*)v_biases);
    QW_HIP_CHECK(hipGetLastError());
    return QW_OK;
}

int KVCache::import_tensors(int n_tokens, const void* k_codes, const void* k_scales,
                            const void* k_biases, const void* v_codes, const void* v_scales,
                            const void* v_biases, hipStream_t stream) {
    QW_REQUIRE(!turbo4(), QW_ERR_STATE, "import: a Turbo4 cache imports with qw_kv_import_turbo4");
    QW_REQUIRE(n_tokens >= 0, QW_ERR_INVALID_ARGUMENT, "import: n_tokens must be >= 0");
    QW_REQUIRE(k_codes && v_codes, QW_ERR_INVALID_ARGUMENT, "import: null code pointers");
    QW_REQUIRE(!affine() || (k_scales && v_scales && (int8() || (k_biases && v_biases))),
               QW_ERR_INVALID_ARGUMENT, "import: null scale/bias pointers");
    DeviceGuard dg(device);
    offset = 0;
    if (n_tokens == 0) return QW_OK;
    if (!affine()) return update(k_codes, v_codes, n_tokens, stream);
    int rc = reserve(n_tokens, stream);
    if (rc) return rc;
    const int n = n_tokens;
    const size_t kr = (size_t)D * bits / 8;
    for (int h = 0; h < hkv; h++)
        QW_HIP_CHECK(hipMemcpyAsync((char*)k_data + h * (size_t)cap * kr,
                                    (const char*)k_codes + h * (size_t)n * kr, n * kr,
                                    hipMemcpyDeviceToDevice, stream));
    // The imported scales decide the fused kernels' dequant path afresh (Int8
    // always takes the separately rounded one).
    hipLaunchKernelGGL(set_flag_kernel, dim3(1), dim3(1), 0, stream, fast_flag, int8() ? 0 : 1);
    const int64_t work = (int64_t)hkv * n * (D * bits / 32);
    const unsigned nb = (unsigned)std::min<int64_t>((work + 255) / 256, 4096);
    if (int8()) {
        hipLaunchKernelGGL(flip_code_sign_kernel, dim3(nb), dim3(256), 0, stream,
                           (uint32_t*)k_data, hkv, n, D / 4, cap);
        QW_HIP_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL(snapshot_affine_kernel, dim3(nb), dim3(256), 0, stream, 1, bits,
                       int8() ? 1 : 0, D, cap, hkv, n, fast_flag, k_params, (uint32_t*)v_data,
                       (f16*)v_params, (f16*)k_scales, (f16*)k_biases, (uint32_t*)v_codes,
                       (f16*)v_scales, (f16*)v_biases);
    QW_HIP_CHECK(hipGetLastError());
    const int64_t vwork = (int64_t)hkv * ((n + 7) / 8) * D;
    hipLaunchKernelGGL(import_v_codes_kernel,
                       dim3((unsigned)std::min<int64_t>((vwork + 255) / 256, 4096)), dim3(256),
                       0, stream, bits, int8() ? 1 : 0, D, cap, hkv, n,
                       (const uint32_t*)v_codes, (uint32_t*)v_data);
    QW_HIP_CHECK(hipGetLastError());
    offset = n;
    return QW_OK;
}

}  // namespace qw
