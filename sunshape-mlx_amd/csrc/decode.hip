// Fused decode: the interleaved-fp16 and bfloat16 matrix-core decodes, the
// prepared codebook, split plans and the bounded waits' failure words.
#include <atomic>
#include <mutex>

#include "decode_host.hpp"

namespace ss {

// Sticky wait-failure word of this code object, one per device (kWait* bits).
__device__ unsigned int g_wait_fail_word;

// Spin limit of the bounded waits for later launches (ss_debug_set_spin_limit).
static std::atomic<int> g_spin_limit{kSpinLimit};

// Pinned host word that a give-up also stores its bits into (one per
// process, mapped into every device): the host polls it after the fact
// with a plain load, so the check costs no synchronisation.
static int wait_host_word(unsigned int **host, unsigned int **dev_ptr) {
    static std::mutex mu;
    static unsigned int *h = nullptr, *d = nullptr;
    std::lock_guard<std::mutex> lock(mu);
    if (!h) {
        void *p = nullptr;
        hipError_t e = hipHostMalloc(&p, 64, hipHostMallocPortable | hipHostMallocMapped |
                                                 hipHostMallocCoherent);
        if (e != hipSuccess) return hip_fail(e, "hipHostMalloc(wait flag)");
        void *dp = nullptr;
        e = hipHostGetDevicePointer(&dp, p, 0);
        if (e != hipSuccess) {
            (void)hipHostFree(p);
            return hip_fail(e, "hipHostGetDevicePointer(wait flag)");
        }
        h = static_cast<unsigned int *>(p);
        *h = 0u;
        d = static_cast<unsigned int *>(dp);
    }
    if (host) *host = h;
    if (dev_ptr) *dev_ptr = d;
    return SS_OK;
}

// Device address of g_wait_fail_word on the current device, looked up once
// per device.
static int wait_word(unsigned int **out) {
    static std::mutex mu;
    static unsigned int *addr[64] = {nullptr};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    SS_UNSUPPORTED(dev >= 0 && dev < 64, "device ordinal %d beyond 63", dev);
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_wait_fail_word));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(wait word)");
        addr[dev] = static_cast<unsigned int *>(p);
    }
    *out = addr[dev];
    return SS_OK;
}

int fill_common(DecodeCommon &c, const DecodeShape &s, const void *q, int q_dtype,
                int hq, int hkv, int64_t t_q, float scale, const int32_t *perm,
                const float *centroids, int n_centroids, const uint8_t *idx, int64_t cap,
                int64_t t_kv, int causal, int64_t q_offset, void *out, int out_dtype,
                void *ws, size_t ws_bytes, int head_dim) {
    c.q = q;
    c.perm = perm;
    c.centroids = centroids;
    c.idx = idx;
    c.out = out;
    c.q_dtype = q_dtype;
    c.out_dtype = out_dtype;
    c.n_q_heads = hq;
    c.n_kv_heads = hkv;
    c.rep = hq / hkv;
    c.n_rg = s.n_rg;
    c.t_q = t_q;
    c.rows_total = (int64_t)c.rep * t_q;
    c.n_centroids = n_centroids;
    c.cap = cap;
    c.t_kv = t_kv;
    c.scale = scale;
    c.causal = causal ? 1 : 0;
    c.q_offset = q_offset;
    c.n_splits = s.S;
    c.tiles_per_split = s.tiles_per_split;
    c.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    {
        int rc = wait_word(&c.wait_fail);
        if (rc == SS_OK) rc = wait_host_word(nullptr, &c.wait_host);
        if (rc != SS_OK) return rc;
    }
    c.kheavy = nullptr;
    c.heavy_dims = nullptr;
    c.nhd = 0;
    c.rot = nullptr;
    c.part_ml = nullptr;
    c.part_acc = nullptr;
    c.part_cnt = nullptr;
    c.fused_merge = s.S > 1 && (size_t)s.n_cols * sizeof(int) <= kCntBytes;
    // columns' counters up to 4 KiB apart, so the splits of different
    // columns never contend for one cache line
    c.cnt_stride = 1024;
    while (c.cnt_stride > 1 && (size_t)s.n_cols * c.cnt_stride * sizeof(int) > kCntBytes)
        c.cnt_stride /= 2;
    if (s.S > 1) {
        const size_t need = decode_ws_bytes(s, head_dim);
        if (!ws || ws_bytes < need) {
            set_error("decode workspace too small: need %zu bytes, got %zu", need,
                      ws ? ws_bytes : (size_t)0);
            return SS_ERR_WORKSPACE;
        }
        SS_REQUIRE(((uintptr_t)ws % 256) == 0, "workspace must be 256-byte aligned");
        const WsLayout w = ws_layout(s, head_dim);
        char *base = reinterpret_cast<char *>(ws);
        c.part_cnt = reinterpret_cast<int *>(base + w.cnt);
        c.part_ml = reinterpret_cast<float *>(base + w.ml);
        c.part_acc = reinterpret_cast<float *>(base + w.acc);
    }
    return SS_OK;
}

}  // namespace ss


using namespace ss;

extern "C" int ss_decode_wait_failures(void *stream, int clear, unsigned int *flags) {
    unsigned int *w = nullptr;
    int rc = wait_word(&w);
    if (rc != SS_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_fail(e, "hipStreamSynchronize");
    unsigned int v = 0;
    e = hipMemcpy(&v, w, sizeof(v), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpy(wait word)");
    unsigned int *hw = nullptr;
    rc = wait_host_word(&hw, nullptr);
    if (rc != SS_OK) return rc;
    v |= __atomic_load_n(hw, __ATOMIC_ACQUIRE);
    if (flags) *flags = v;
    if (v && clear) {
        const unsigned int zero = 0;
        e = hipMemcpy(w, &zero, sizeof(zero), hipMemcpyHostToDevice);
        if (e != hipSuccess) return hip_fail(e, "hipMemcpy(clear wait word)");
        __atomic_store_n(hw, 0u, __ATOMIC_RELEASE);
    }
    if (v) {
        set_error("a bounded wait of a fused decode gave up (flags 0x%x: %s%s%s); the output of "
                  "that launch is invalid", v, (v & kWaitBarrier) ? "compute barrier " : "",
                  (v & kWaitSlot) ? "ring slot " : "", (v & kWaitTile) ? "ring tile" : "");
        return SS_ERR_WAIT;
    }
    return SS_OK;
}

extern "C" int ss_decode_wait_flag_host(unsigned int **flag) {
    SS_REQUIRE(flag, "null pointer argument");
    return wait_host_word(flag, nullptr);
}

extern "C" int ss_debug_set_spin_limit(int limit) {
    g_spin_limit.store(limit < 0 ? kSpinLimit : limit, std::memory_order_relaxed);
    return SS_OK;
}

extern "C" size_t ss_decode_workspace_bytes(int64_t batch, int n_q_heads, int n_kv_heads,
                                            int64_t t_q, int head_dim, int64_t t_kv,
                                            int n_splits) {
    if (batch < 1 || n_q_heads < 1 || n_kv_heads < 1 || n_q_heads % n_kv_heads || t_q < 1)
        return 0;
    return decode_ws_bytes(decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits),
                           head_dim);
}

extern "C" int ss_decode_default_splits(int64_t batch, int n_q_heads, int n_kv_heads,
                                        int64_t t_q, int head_dim, int64_t t_kv) {
    (void)head_dim;
    if (batch < 1 || n_q_heads < 1 || n_kv_heads < 1 || n_q_heads % n_kv_heads || t_q < 1)
        return 0;
    return decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, 0).S;
}

extern "C" size_t ss_decode_turboquant_workspace_bytes(int64_t batch, int n_q_heads,
                                                       int n_kv_heads, int64_t t_q, int head_dim,
                                                       int64_t t_kv, int64_t t_buf, int n_splits) {
    if (batch < 1 || n_q_heads < 1 || n_kv_heads < 1 || n_q_heads % n_kv_heads || t_q < 1)
        return 0;
    // enough for every split policy of the transformed-basis decodes (the
    // VALU kernel's, the matrix-core TurboQuant and SunShape-value kernels')
    size_t need = 0;
    for (int kind : {kKindValu, kKindMfma, kKindSunv}) {
        const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits, kind);
        need = std::max(need, turboquant_ws_bytes(with_buffer_slot(s, t_buf), batch * n_q_heads * t_q,
                                                  head_dim));
    }
    return need;
}

extern "C" int ss_decode_plan(int kind, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
                              int head_dim, int64_t t_kv, int n_splits, int *splits_out,
                              size_t *workspace_bytes_out) {
    SS_REQUIRE(kind == kKindValu || kind == kKindMfma, "kind must be 0 (dense) or 1 (il8)");
    SS_REQUIRE(batch >= 1 && n_q_heads >= 1 && n_kv_heads >= 1 && t_q >= 1 &&
                   n_q_heads % n_kv_heads == 0,
               "bad head/batch counts");
    const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits, kind);
    if (splits_out) *splits_out = s.S;
    if (workspace_bytes_out) *workspace_bytes_out = decode_ws_bytes(s, head_dim);
    return SS_OK;
}

// One workgroup: max |C| over the codebook, then C' = C * 2^(kCbMaxExp - e)
// (max |C| < 2^e) split into fp16 hi/lo, stored in the order the LUT build's
// matrix-core operands are loaded: tile (bg, ct) of 4 blocks x 16 centroids
// holds 64 lanes x 8 halves for hi, then the same for lo, where lane l
// carries centroid ct*16 + l%16 of block bg*4 + l/16 (zero past the last
// centroid).  The multiplier 2^(e - kCbMaxExp) that undoes the scale follows
// as a float.
__global__ void __launch_bounds__(1024) codebook_f16x2_kernel(const float *cents, int n_blocks,
                                                              int n_centroids, _Float16 *out) {
    __shared__ float red[1024 / kWave];
    const int n = n_blocks * n_centroids * kBlockDim;
    float mx = 0.f;
    for (int i = threadIdx.x; i < n; i += 1024) mx = fmaxf(mx, fabsf(cents[i]));
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int w = 1; w < 1024 / kWave; ++w) mx = fmaxf(mx, red[w]);
    int ex = 0;
    frexpf(mx, &ex);  // mx < 2^ex
    const int sh = kCbMaxExp - ex;
    const int nct = (n_centroids + 15) / 16;
    const int n_lanes = cb_tiles(n_blocks, n_centroids) * kWave;
    for (int i = threadIdx.x; i < n_lanes * kBlockDim; i += 1024) {
        const int j = i % kBlockDim, lane = (i / kBlockDim) % kWave, tile = i / (kBlockDim * kWave);
        const int bg = tile / nct, ct = tile % nct;
        const int b = bg * 4 + lane / 16, cc = ct * 16 + lane % 16;
        const float v = cc < n_centroids
                            ? ldexpf(cents[((int64_t)b * n_centroids + cc) * kBlockDim + j], sh)
                            : 0.f;
        const _Float16 hi = (_Float16)v;
        _Float16 *o = out + (int64_t)tile * 2 * kWave * kBlockDim + lane * kBlockDim + j;
        o[0] = hi;
        o[kWave * kBlockDim] = (_Float16)((v - (float)hi) * kSplitScale);
    }
    if (threadIdx.x == 0)
        *reinterpret_cast<float *>(out + (int64_t)n_lanes * 2 * kBlockDim) = ldexpf(1.f, -sh);
    // |C|^2 of each lane's centroid (unscaled float32, 0 past the last
    // centroid), in the tiles' lane order, after the scale's 16 bytes
    float *nrm = reinterpret_cast<float *>(out + (int64_t)n_lanes * 2 * kBlockDim) + 4;
    for (int i = threadIdx.x; i < n_lanes; i += 1024) {
        const int lane = i % kWave, tile = i / kWave;
        const int bg = tile / nct, ct = tile % nct;
        const int b = bg * 4 + lane / 16, cc = ct * 16 + lane % 16;
        float acc = 0.f;
        if (cc < n_centroids)
            for (int j = 0; j < kBlockDim; ++j) {
                const float x = cents[((int64_t)b * n_centroids + cc) * kBlockDim + j];
                acc = fmaf(x, x, acc);
            }
        nrm[i] = acc;
    }
}

extern "C" size_t ss_codebook_f16x2_bytes(int n_blocks, int n_centroids) {
    if (n_blocks < 4 || n_blocks % 4 || n_centroids < 1) return 0;
    return (size_t)cb_tiles(n_blocks, n_centroids) * kWave * (2 * 16 + 4) + 16;
}

extern "C" int ss_codebook_f16x2(const float *centroids, int n_blocks, int n_centroids,
                                 void *out, void *stream) {
    SS_REQUIRE(centroids && out, "null centroids/out");
    SS_REQUIRE(n_blocks >= 4 && n_blocks <= 64 && n_blocks % 4 == 0 && n_centroids >= 1 &&
                   n_centroids <= kLutStride,
               "bad codebook shape (%d blocks, %d centroids)", n_blocks, n_centroids);
    SS_REQUIRE(((uintptr_t)out % 16) == 0, "prepared codebook must be 16-byte aligned");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(codebook_f16x2_kernel, dim3(1), dim3(1024), 0, st, centroids, n_blocks,
                       n_centroids, static_cast<_Float16 *>(out));
    SS_LAUNCH_CHECK("codebook_f16x2_kernel launch");
    return SS_OK;
}

static int il8_impl(const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads,
                    int64_t t_q, int head_dim, float scale, const int32_t *perm,
                    const void *codebook, int n_blocks, int n_centroids, const uint8_t *idx,
                    const void *values_il8, int v_dtype, int64_t cap, int64_t t_kv, int causal,
                    int64_t q_offset, void *out, int out_dtype, void *workspace,
                    size_t workspace_bytes, int n_splits, const void *k_buf, const void *v_buf,
                    int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st,
                    int64_t t_buf, void *stream, const void *k_heavy = nullptr,
                    const int32_t *heavy_dims = nullptr, int n_heavy_dims = 0,
                    const ss_attn_mask *mask = nullptr) {
    const float *cents = static_cast<const float *>(codebook);
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, cents,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    SS_REQUIRE(((uintptr_t)codebook % 16) == 0, "prepared codebook must be 16-byte aligned");
    SS_REQUIRE(values_il8, "null values");
    SS_UNSUPPORTED(v_dtype == SS_F16, "interleaved values must be float16");
    SS_REQUIRE(cap % 8 == 0, "cap must be a multiple of 8 for interleaved values");
    SS_REQUIRE(((uintptr_t)values_il8 % 16) == 0, "values must be 16-byte aligned");
    const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits,
                                       kKindMfma);
    DecodeCommon c;
    rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, cents,
                     n_centroids, idx, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                     workspace_bytes, head_dim);
    if (rc) return rc;
    c.centroids = nullptr;
    c.codebook = static_cast<const uint4 *>(codebook);
    c.codebook_mul = reinterpret_cast<const float *>(
        static_cast<const char *>(codebook) + (size_t)cb_tiles(n_blocks, n_centroids) * 2 * kWave * 16);
    rc = check_buffer(k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf, head_dim);
    if (rc) return rc;
    rc = set_heavy(c, k_heavy, heavy_dims, n_heavy_dims);
    if (rc) return rc;
    if ((rc = set_mask(c, mask))) return rc;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const __half *v8 = reinterpret_cast<const __half *>(values_il8);
    // the hybrid cache's kernel (buffer share, heavy dims, masks)
    if (t_buf > 0 || c.nhd > 0 || c.mask_dt != kMaskNone) {
        if (head_dim == 128)
            return launch_mfma<128, VIl8Hyb<128>>(
                c, VIl8Hyb<128>::Args{v8, k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf},
                s, st);
        return launch_mfma<64, VIl8Hyb<64>>(
            c, VIl8Hyb<64>::Args{v8, k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf}, s,
            st);
    }
    if (head_dim == 128) return launch_mfma<128, VIl8<128>>(c, VIl8<128>::Args{v8}, s, st);
    return launch_mfma<64, VIl8<64>>(c, VIl8<64>::Args{v8}, s, st);
}

extern "C" int ss_decode_attn_il8(const void *q, int q_dtype, int64_t batch, int n_q_heads,
                                  int n_kv_heads, int64_t t_q, int head_dim, float scale,
                                  const int32_t *perm, const void *codebook, int n_blocks,
                                  int n_centroids, const uint8_t *idx, const void *values_il8,
                                  int v_dtype, int64_t cap, int64_t t_kv, int causal,
                                  int64_t q_offset, void *out, int out_dtype, void *workspace,
                                  size_t workspace_bytes, int n_splits, void *stream) {
    return il8_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                    codebook, n_blocks, n_centroids, idx, values_il8, v_dtype, cap, t_kv, causal,
                    q_offset, out, out_dtype, workspace, workspace_bytes, n_splits, nullptr,
                    nullptr, SS_F16, 0, 0, 0, 0, stream);
}

extern "C" int ss_decode_attn_il8_hybrid(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values_il8, int v_dtype, int64_t cap,
    int64_t t_kv, const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb,
    int64_t buf_sh, int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims,
    int n_heavy_dims, int causal, int64_t q_offset, void *out, int out_dtype, void *workspace,
    size_t workspace_bytes, int n_splits, void *stream) {
    return il8_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                    codebook, n_blocks, n_centroids, idx, values_il8, v_dtype, cap, t_kv, causal,
                    q_offset, out, out_dtype, workspace, workspace_bytes, n_splits, k_buf, v_buf,
                    buf_dtype, buf_sb, buf_sh, buf_st, t_buf, stream, k_heavy, heavy_dims,
                    n_heavy_dims);
}

extern "C" int ss_decode_attn_il8_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values_il8, int v_dtype, int64_t cap,
    int64_t t_kv, const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb,
    int64_t buf_sh, int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims,
    int n_heavy_dims, int causal, int64_t q_offset, void *out, int out_dtype, void *workspace,
    size_t workspace_bytes, int n_splits, const ss_attn_mask *mask, void *stream) {
    return il8_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                    codebook, n_blocks, n_centroids, idx, values_il8, v_dtype, cap, t_kv, causal,
                    q_offset, out, out_dtype, workspace, workspace_bytes, n_splits, k_buf, v_buf,
                    buf_dtype, buf_sb, buf_sh, buf_st, t_buf, stream, k_heavy, heavy_dims,
                    n_heavy_dims, mask);
}

static int decode_attn_dense_mfma_impl(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values, int v_dtype, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    const float *cents = static_cast<const float *>(codebook);
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, cents,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    if ((rc = dense_checks(values, v_dtype))) return rc;
    SS_UNSUPPORTED(v_dtype == SS_BF16, "the matrix-core dense decode takes bfloat16 values");
    const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits,
                                       kKindMfma);
    DecodeCommon c;
    rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, cents,
                     n_centroids, idx, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                     workspace_bytes, head_dim);
    if (rc) return rc;
    c.centroids = nullptr;
    c.codebook = static_cast<const uint4 *>(codebook);
    c.codebook_mul = reinterpret_cast<const float *>(
        static_cast<const char *>(codebook) + (size_t)cb_tiles(n_blocks, n_centroids) * 2 * kWave * 16);
    rc = check_buffer(k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf, head_dim);
    if (rc) return rc;
    if ((rc = set_heavy(c, k_heavy, heavy_dims, n_heavy_dims))) return rc;
    if ((rc = set_mask(c, mask))) return rc;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const __hip_bfloat16 *v = static_cast<const __hip_bfloat16 *>(values);
    if (head_dim == 128)
        return launch_mfma<128, VBf16<128>>(
            c, VBf16<128>::Args{v, k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf}, s, st);
    return launch_mfma<64, VBf16<64>>(
        c, VBf16<64>::Args{v, k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf}, s, st);
}

extern "C" int ss_decode_attn_dense_mfma(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values, int v_dtype, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, void *stream) {
    return decode_attn_dense_mfma_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                       scale, perm, codebook, n_blocks, n_centroids, idx, values,
                                       v_dtype, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb, buf_sh,
                                       buf_st, t_buf, k_heavy, heavy_dims, n_heavy_dims, causal,
                                       q_offset, out, out_dtype, workspace, workspace_bytes,
                                       n_splits, nullptr, stream);
}

extern "C" int ss_decode_attn_dense_mfma_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values, int v_dtype, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    return decode_attn_dense_mfma_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                       scale, perm, codebook, n_blocks, n_centroids, idx, values,
                                       v_dtype, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb, buf_sh,
                                       buf_st, t_buf, k_heavy, heavy_dims, n_heavy_dims, causal,
                                       q_offset, out, out_dtype, workspace, workspace_bytes,
                                       n_splits, mask, stream);
}

// ---------------------------------------------------------------------------
// Allocation-free variant of ss_decode_attn_il8.  Its split partials and
// per-column counters live in a file-scope device array (one per GPU, held
// until the process ends) instead of a caller workspace.  Host code never
// uses the array's name as an address: the per-device address comes from
// hipGetSymbolAddress at the first call on each device, which also clears
// the counter area with a fill kernel; every completed call leaves it zero.
// ---------------------------------------------------------------------------
constexpr size_t kStaticScratchBytes = 4u << 20;  // 4 MiB per device
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

__global__ void __launch_bounds__(256) zero_words_kernel(uint32_t *p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

// Device address of `scratch` on the current device, looked up (and its
// counter area cleared on `st`) at the first call on that device.
static int static_scratch(void **out, hipStream_t st) {
    static std::mutex mu;
    static void *addr[64] = {nullptr};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    SS_UNSUPPORTED(dev >= 0 && dev < 64, "device ordinal %d beyond 63", dev);
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        hipLaunchKernelGGL(zero_words_kernel, dim3(64), dim3(256), 0, st,
                           static_cast<uint32_t *>(p), (int64_t)(kCntBytes / 4));
        SS_LAUNCH_CHECK("zero_words_kernel launch");
        addr[dev] = p;
    }
    *out = addr[dev];
    return SS_OK;
}

extern "C" size_t ss_decode_static_scratch_bytes(void) { return kStaticScratchBytes; }

extern "C" int ss_decode_attn_il8_noalloc(const void *q, int q_dtype, int64_t batch,
                                          int n_q_heads, int n_kv_heads, int64_t t_q,
                                          int head_dim, float scale, const int32_t *perm,
                                          const void *codebook, int n_blocks, int n_centroids,
                                          const uint8_t *idx, const void *values_il8,
                                          int v_dtype, int64_t cap, int64_t t_kv, int causal,
                                          int64_t q_offset, void *out, int out_dtype,
                                          int n_splits, void *stream) {
    SS_REQUIRE(batch >= 1 && n_q_heads >= 1 && n_kv_heads >= 1 && t_q >= 1 &&
                   n_q_heads % n_kv_heads == 0,
               "bad head/batch counts");
    SS_UNSUPPORTED(head_dim == 64 || head_dim == 128, "head_dim %d unsupported (64 or 128)",
                   head_dim);
    const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits,
                                       kKindMfma);
    const size_t need = decode_ws_bytes(s, head_dim);
    if (need > kStaticScratchBytes) {
        set_error("ss_decode_attn_il8_noalloc: this shape needs %zu bytes of split scratch "
                  "(%d splits), the static scratch holds %zu; pass fewer splits or use "
                  "ss_decode_attn_il8 with a workspace",
                  need, s.S, kStaticScratchBytes);
        return SS_ERR_WORKSPACE;
    }
    void *ws = nullptr;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (need > 0) {
        const int rc = static_scratch(&ws, st);
        if (rc) return rc;
    }
    return ss_decode_attn_il8(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale,
                              perm, codebook, n_blocks, n_centroids, idx, values_il8, v_dtype,
                              cap, t_kv, causal, q_offset, out, out_dtype, ws,
                              need > 0 ? kStaticScratchBytes : 0, n_splits, stream);
}
