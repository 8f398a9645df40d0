// Decode steps that append their tokens and attend in one launch.
#include "decode_host.hpp"

using namespace ss;

extern "C" int ss_decode_step_il8(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, const float *centroids,
    int n_blocks, int n_centroids, uint8_t *idx, void *values_il8, int64_t cap, int64_t t_cache,
    const void *k_new, const void *v_new, int kv_dtype, int64_t kv_sb, int64_t kv_sh, int64_t kv_st,
    int64_t n_new, int causal, int64_t q_offset, void *out, int out_dtype, void *workspace,
    size_t workspace_bytes, int n_splits, void *stream) {
    SS_UNSUPPORTED(n_new >= 1 && n_new <= kMaxStepTokens, "a fused step takes 1..%d new tokens",
                   kMaxStepTokens);
    SS_REQUIRE(t_cache >= 1, "a fused step needs a non-empty cache (t_cache %lld)",
               (long long)t_cache);
    SS_REQUIRE(t_cache + n_new <= cap, "new tokens [%lld, %lld) past cap %lld", (long long)t_cache,
               (long long)(t_cache + n_new), (long long)cap);
    SS_UNSUPPORTED(kv_dtype == SS_F16, "a fused step takes float16 keys and values");
    SS_REQUIRE(k_new && v_new && centroids, "null new keys, values or centroids");
    SS_UNSUPPORTED(n_centroids >= 1 && n_centroids <= 256 && n_blocks * 8 == head_dim,
                   "a fused step needs 8-dim blocks of at most 256 centroids");
    const float *cents = static_cast<const float *>(codebook);
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, cents,
                          n_blocks, n_centroids, idx, cap, t_cache, out, out_dtype);
    if (rc) return rc;
    SS_REQUIRE(((uintptr_t)codebook % 16) == 0, "prepared codebook must be 16-byte aligned");
    SS_REQUIRE(((uintptr_t)centroids % 16) == 0, "centroids must be 16-byte aligned");
    SS_REQUIRE(values_il8, "null values");
    SS_REQUIRE(cap % 8 == 0, "cap must be a multiple of 8 for interleaved values");
    SS_REQUIRE(((uintptr_t)values_il8 % 16) == 0, "values must be 16-byte aligned");
    rc = check_buffer(k_new, v_new, kv_dtype, kv_sb, kv_sh, kv_st, n_new, head_dim);
    if (rc) return rc;
    const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_cache, n_splits,
                                       kKindMfma);
    DecodeCommon c;
    rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, cents,
                     n_centroids, idx, cap, t_cache, causal, q_offset, out, out_dtype, workspace,
                     workspace_bytes, head_dim);
    if (rc) return rc;
    c.centroids = nullptr;
    c.codebook = static_cast<const uint4 *>(codebook);
    c.codebook_mul = reinterpret_cast<const float *>(
        static_cast<const char *>(codebook) + (size_t)cb_tiles(n_blocks, n_centroids) * 2 * kWave * 16);
    if (s.S > 1) {
        // the last split encodes and attends the new tokens before its tiles:
        // it gives up about kStepShareTokens cache tokens to the others, 8 at
        // a time, as far as its own range allows
        const int64_t room = t_cache - (int64_t)(s.S - 1) * s.tiles_per_split * kWave;
        const int64_t want = (kStepShareTokens + (s.S - 1) * 8 - 1) / ((int64_t)(s.S - 1) * 8) * 8;
        const int64_t most = room > 0 ? room / (s.S - 1) / 8 * 8 : 0;
        c.split_pad = (int)(want < most ? want : most);
    }
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    __half *v8 = reinterpret_cast<__half *>(values_il8);
    const float *norms = c.codebook_mul + 4;
    if (head_dim == 128)
        return launch_mfma<128, VIl8Step<128>>(
            c, VIl8Step<128>::Args{v8, k_new, v_new, kv_dtype, kv_sb, kv_sh, kv_st, n_new, centroids,
                                   norms, idx, v8},
            s, st);
    return launch_mfma<64, VIl8Step<64>>(
        c, VIl8Step<64>::Args{v8, k_new, v_new, kv_dtype, kv_sb, kv_sh, kv_st, n_new, centroids, norms,
                              idx, v8},
        s, st);
}

// The checks and launch set-up shared by the hybrid-step entry points:
// step sizes, the buffer window and the new tokens, then the common decode
// arguments and the last split's hand-over of cache tokens.
static int hybrid_step_setup(DecodeCommon &c, DecodeShape &s, const void *q, int q_dtype,
                             int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
                             int head_dim, float scale, const int32_t *perm, const void *codebook,
                             const float *centroids, int n_blocks, int n_centroids,
                             const uint8_t *idx, int64_t cap, int64_t t_kv, const void *k_buf,
                             const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
                             int64_t buf_st, int64_t n_buf, int64_t n_flush, const void *k_new,
                             const void *v_new, int kv_dtype, int64_t kv_sb, int64_t kv_sh,
                             int64_t kv_st, int64_t n_new, int causal, int64_t q_offset, void *out,
                             int out_dtype, void *workspace, size_t workspace_bytes, int n_splits,
                             int pad_unit) {
    SS_UNSUPPORTED(n_new >= 1 && n_new <= kMaxStepTokens, "a fused step takes 1..%d new tokens",
                   kMaxStepTokens);
    SS_UNSUPPORTED(n_flush >= 0 && n_flush <= kMaxStepTokens,
                   "a fused hybrid step flushes 0..%d tokens (got %lld)", kMaxStepTokens,
                   (long long)n_flush);
    SS_REQUIRE(n_buf >= n_flush, "n_flush %lld exceeds the %lld buffered tokens", (long long)n_flush,
               (long long)n_buf);
    SS_REQUIRE(t_kv >= 1, "a fused hybrid step needs compressed tokens (t_kv %lld)", (long long)t_kv);
    SS_REQUIRE(t_kv + n_flush <= cap, "flushed tokens [%lld, %lld) past cap %lld", (long long)t_kv,
               (long long)(t_kv + n_flush), (long long)cap);
    SS_UNSUPPORTED(kv_dtype == SS_F16 && buf_dtype == SS_F16,
                   "a fused hybrid step takes a float16 buffer and float16 new tokens");
    SS_REQUIRE(k_new && v_new && centroids, "null new keys, values or centroids");
    SS_REQUIRE(((uintptr_t)codebook % 16) == 0, "prepared codebook must be 16-byte aligned");
    const float *cents = static_cast<const float *>(codebook);
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, centroids,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    // buffer rows 0 .. n_buf + n_new - 1 are read or written
    rc = check_buffer(k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, n_buf + n_new, head_dim);
    if (rc) return rc;
    rc = check_buffer(k_new, v_new, kv_dtype, kv_sb, kv_sh, kv_st, n_new, head_dim);
    if (rc) return rc;
    s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits, kKindMfma);
    rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, cents,
                     n_centroids, idx, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                     workspace_bytes, head_dim);
    if (rc) return rc;
    c.centroids = nullptr;
    c.codebook = static_cast<const uint4 *>(codebook);
    c.codebook_mul = reinterpret_cast<const float *>(
        static_cast<const char *>(codebook) + (size_t)cb_tiles(n_blocks, n_centroids) * 2 * kWave * 16);
    if (s.S > 1 && n_flush > 0) {
        // the last split encodes and attends the flushed tokens before its
        // tiles: it gives up some cache tokens to the others, in units of
        // pad_unit tokens (a split must start on a code word: 64 for grouped
        // codes, whose 2-bit words hold 16 tokens; 8 for interleaved fp16)
        const int64_t pu = pad_unit;
        const int64_t room = t_kv - (int64_t)(s.S - 1) * s.tiles_per_split * kWave;
        const int64_t want = (kHybridStepShareTokens + (s.S - 1) * pu - 1) / ((int64_t)(s.S - 1) * pu) * pu;
        const int64_t most = room > 0 ? room / (s.S - 1) / pu * pu : 0;
        c.split_pad = (int)(want < most ? want : most);
    }
    return SS_OK;
}

extern "C" int ss_decode_step_grouped_il_hybrid(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, const float *centroids,
    int n_blocks, int n_centroids, uint8_t *idx, uint32_t *codes_il, void *scales, void *zeros,
    int sz_dtype, int bits, int group_size, int64_t cap, int64_t t_kv, void *k_buf, void *v_buf,
    int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t n_buf, int64_t n_flush,
    const void *k_new, const void *v_new, int kv_dtype, int64_t kv_sb, int64_t kv_sh, int64_t kv_st,
    int64_t n_new, int causal, int64_t q_offset, void *out, int out_dtype, void *workspace,
    size_t workspace_bytes, int n_splits, void *stream) {
    SS_REQUIRE(codes_il && scales && zeros, "null codes, scales or zeros");
    SS_UNSUPPORTED(bits == 2 || bits == 4, "a fused hybrid step takes 2- or 4-bit codes (got %d)",
                   bits);
    SS_UNSUPPORTED(group_size == head_dim || 2 * group_size == head_dim,
                   "group_size %d: the fused kernel takes one or two groups per row", group_size);
    SS_REQUIRE(sz_dtype == SS_F32 || sz_dtype == SS_F16, "scale/zero dtype must be f32 or f16");
    SS_REQUIRE(cap % 16 == 0, "cap must be a multiple of 16 for interleaved grouped values");
    SS_REQUIRE(((uintptr_t)codes_il % 16) == 0 && ((uintptr_t)scales % 16) == 0 &&
                   ((uintptr_t)zeros % 16) == 0,
               "codes, scales and zeros must be 16-byte aligned");
    DecodeCommon c;
    DecodeShape s;
    int rc = hybrid_step_setup(c, s, q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale,
                               perm, codebook, centroids, n_blocks, n_centroids, idx, cap, t_kv,
                               k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, n_buf, n_flush,
                               k_new, v_new, kv_dtype, kv_sb, kv_sh, kv_st, n_new, causal, q_offset,
                               out, out_dtype, workspace, workspace_bytes, n_splits, kWave);
    if (rc) return rc;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const float *norms = c.codebook_mul + 4;
    const int ng = head_dim / group_size;
#define SS_GSTEP(DD, BB, NGG, SZT)                                                              \
    {                                                                                           \
        using VF = VGilStep<DD, BB, NGG, SZT>;                                                  \
        typename VF::Args a{};                                                                  \
        a.codes = codes_il;                                                                     \
        a.scales = static_cast<const SZT *>(scales);                                            \
        a.zeros = static_cast<const SZT *>(zeros);                                              \
        a.kbuf = k_buf;                                                                         \
        a.vbuf = v_buf;                                                                         \
        a.buf_dtype = buf_dtype;                                                                \
        a.buf_sb = buf_sb;                                                                      \
        a.buf_sh = buf_sh;                                                                      \
        a.buf_st = buf_st;                                                                      \
        a.t_buf = n_buf - n_flush + n_new;                                                      \
        a.knew = k_new;                                                                         \
        a.vnew = v_new;                                                                         \
        a.new_sb = kv_sb;                                                                       \
        a.new_sh = kv_sh;                                                                       \
        a.new_st = kv_st;                                                                       \
        a.n_rem = n_buf - n_flush;                                                              \
        a.n_flush = n_flush;                                                                    \
        a.centroids = centroids;                                                                \
        a.cb_norms = norms;                                                                     \
        a.idx_out = idx;                                                                        \
        a.codes_out = codes_il;                                                                 \
        a.scales_out = static_cast<SZT *>(scales);                                              \
        a.zeros_out = static_cast<SZT *>(zeros);                                                \
        a.kput = k_buf;                                                                         \
        a.vput = v_buf;                                                                         \
        return launch_mfma<DD, VF>(c, a, s, st);                                                \
    }
#define SS_GSTEP_SZ(DD, BB, NGG)                             \
    {                                                        \
        if (sz_dtype == SS_F16) SS_GSTEP(DD, BB, NGG, __half) \
        SS_GSTEP(DD, BB, NGG, float)                         \
    }
#define SS_GSTEP_NG(DD, BB)                  \
    {                                        \
        if (ng == 2) SS_GSTEP_SZ(DD, BB, 2)  \
        SS_GSTEP_SZ(DD, BB, 1)               \
    }
    if (head_dim == 128) {
        if (bits == 2) SS_GSTEP_NG(128, 2)
        SS_GSTEP_NG(128, 4)
    }
    if (bits == 2) SS_GSTEP_NG(64, 2)
    SS_GSTEP_NG(64, 4)
#undef SS_GSTEP_NG
#undef SS_GSTEP_SZ
#undef SS_GSTEP
}

extern "C" int ss_decode_step_il8_hybrid(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, const float *centroids,
    int n_blocks, int n_centroids, uint8_t *idx, void *values_il8, int64_t cap, int64_t t_kv,
    void *k_buf, void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st,
    int64_t n_buf, int64_t n_flush, const void *k_new, const void *v_new, int kv_dtype,
    int64_t kv_sb, int64_t kv_sh, int64_t kv_st, int64_t n_new, int causal, int64_t q_offset,
    void *out, int out_dtype, void *workspace, size_t workspace_bytes, int n_splits, void *stream) {
    SS_REQUIRE(values_il8, "null values");
    SS_REQUIRE(cap % 8 == 0, "cap must be a multiple of 8 for interleaved values");
    SS_REQUIRE(((uintptr_t)values_il8 % 16) == 0, "values must be 16-byte aligned");
    DecodeCommon c;
    DecodeShape s;
    int rc = hybrid_step_setup(c, s, q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale,
                               perm, codebook, centroids, n_blocks, n_centroids, idx, cap, t_kv,
                               k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, n_buf, n_flush,
                               k_new, v_new, kv_dtype, kv_sb, kv_sh, kv_st, n_new, causal, q_offset,
                               out, out_dtype, workspace, workspace_bytes, n_splits, 8);
    if (rc) return rc;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const float *norms = c.codebook_mul + 4;
    __half *v8 = static_cast<__half *>(values_il8);
    auto run = [&](auto dtag) {
        constexpr int DD = decltype(dtag)::value;
        using VF = VIl8HybStep<DD>;
        typename VF::Args a{};
        a.v8 = v8;
        a.kbuf = k_buf;
        a.vbuf = v_buf;
        a.buf_dtype = buf_dtype;
        a.buf_sb = buf_sb;
        a.buf_sh = buf_sh;
        a.buf_st = buf_st;
        a.t_buf = n_buf - n_flush + n_new;
        a.knew = k_new;
        a.vnew = v_new;
        a.new_sb = kv_sb;
        a.new_sh = kv_sh;
        a.new_st = kv_st;
        a.n_rem = n_buf - n_flush;
        a.n_flush = n_flush;
        a.centroids = centroids;
        a.cb_norms = norms;
        a.idx_out = idx;
        a.v8_out = v8;
        a.kput = k_buf;
        a.vput = v_buf;
        return launch_mfma<DD, VF>(c, a, s, st);
    };
    if (head_dim == 128) return run(std::integral_constant<int, 128>{});
    return run(std::integral_constant<int, 64>{});
}
