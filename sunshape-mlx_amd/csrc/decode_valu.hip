// Fused decode on the vector ALUs (any value dtype, reference-format grouped
// and TurboQuant values) and of SunShape-coded values.
#include "decode_host.hpp"

using namespace ss;

// The VALU decode over dense values (merge: whether it launches its own merge).
static int launch_dense(const DecodeCommon &c, const DecodeShape &s, hipStream_t st, int head_dim,
                        const void *values, int v_dtype, bool merge) {
#define SS_DENSE(DD, TT)                                                                  \
    {                                                                                     \
        typename VDense<DD, TT>::Args va{reinterpret_cast<const TT *>(values)};           \
        return launch_r<DD, VDense<DD, TT>>(c, va, s, st, merge);                         \
    }
    if (head_dim == 128) {
        if (v_dtype == SS_F16) SS_DENSE(128, __half)
        if (v_dtype == SS_BF16) SS_DENSE(128, __hip_bfloat16)
        SS_DENSE(128, float)
    } else {
        if (v_dtype == SS_F16) SS_DENSE(64, __half)
        if (v_dtype == SS_BF16) SS_DENSE(64, __hip_bfloat16)
        SS_DENSE(64, float)
    }
#undef SS_DENSE
}

extern "C" int ss_decode_attn_dense(const void *q, int q_dtype, int64_t batch, int n_q_heads,
                                    int n_kv_heads, int64_t t_q, int head_dim, float scale,
                                    const int32_t *perm, const float *centroids, int n_blocks,
                                    int n_centroids, const uint8_t *idx, const void *values,
                                    int v_dtype, int64_t cap, int64_t t_kv, int causal,
                                    int64_t q_offset, void *out, int out_dtype, void *workspace,
                                    size_t workspace_bytes, int n_splits, void *stream) {
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, centroids,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    if ((rc = dense_checks(values, v_dtype))) return rc;
    const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits);
    DecodeCommon c;
    rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, centroids,
                     n_centroids, idx, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                     workspace_bytes, head_dim);
    if (rc) return rc;
    return launch_dense(c, s, reinterpret_cast<hipStream_t>(stream), head_dim, values, v_dtype,
                        true);
}

// The VALU decode over reference-format grouped values (merge: whether it
// launches its own merge).
static int launch_grouped(const DecodeCommon &c, const DecodeShape &s, hipStream_t st,
                          int head_dim, const uint32_t *packed, const void *scales,
                          const void *zeros, int sz_dtype, int bits, int group_size, bool merge) {
    const int n_groups = head_dim / group_size;
#define SS_GROUPED(DD, BB, SZT)                                                          \
    {                                                                                    \
        typename VGrouped<DD, BB, SZT>::Args va{packed, reinterpret_cast<const SZT *>(scales), \
                                                reinterpret_cast<const SZT *>(zeros),    \
                                                group_size, n_groups};                   \
        return launch_r<DD, VGrouped<DD, BB, SZT>>(c, va, s, st, merge);                 \
    }
#define SS_GROUPED_BITS(DD, SZT)            \
    {                                       \
        if (bits == 2) SS_GROUPED(DD, 2, SZT) \
        if (bits == 3) SS_GROUPED(DD, 3, SZT) \
        SS_GROUPED(DD, 4, SZT)              \
    }
    if (head_dim == 128) {
        if (sz_dtype == SS_F16) SS_GROUPED_BITS(128, __half)
        SS_GROUPED_BITS(128, float)
    } else {
        if (sz_dtype == SS_F16) SS_GROUPED_BITS(64, __half)
        SS_GROUPED_BITS(64, float)
    }
#undef SS_GROUPED_BITS
#undef SS_GROUPED
}

extern "C" int ss_decode_attn_grouped(const void *q, int q_dtype, int64_t batch, int n_q_heads,
                                      int n_kv_heads, int64_t t_q, int head_dim, float scale,
                                      const int32_t *perm, const float *centroids, int n_blocks,
                                      int n_centroids, const uint8_t *idx,
                                      const uint32_t *packed, const void *scales,
                                      const void *zeros, int sz_dtype, int bits,
                                      int group_size, int64_t cap, int64_t t_kv, int causal,
                                      int64_t q_offset, void *out, int out_dtype, void *workspace,
                                      size_t workspace_bytes, int n_splits, void *stream) {
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, centroids,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    if ((rc = grouped_checks(head_dim, packed, scales, zeros, sz_dtype, bits, group_size)))
        return rc;
    const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits);
    DecodeCommon c;
    rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, centroids,
                     n_centroids, idx, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                     workspace_bytes, head_dim);
    if (rc) return rc;
    return launch_grouped(c, s, reinterpret_cast<hipStream_t>(stream), head_dim, packed, scales,
                          zeros, sz_dtype, bits, group_size, true);
}

static int decode_attn_turboquant_impl(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const float *norms,
    const float *levels, const float *rotation, int bits, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, centroids,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    SS_REQUIRE(packed && norms && levels && rotation, "null packed/norms/levels/rotation");
    if (k_heavy) {
        SS_REQUIRE(heavy_dims, "null heavy_dims");
        SS_UNSUPPORTED(n_heavy_dims > 0 && n_heavy_dims % 8 == 0 && n_heavy_dims <= 64,
                       "n_heavy_dims %d unsupported (a positive multiple of 8, at most 64)",
                       n_heavy_dims);
        SS_REQUIRE(((uintptr_t)k_heavy % 16) == 0, "heavy keys must be 16-byte aligned");
    }
    SS_REQUIRE(bits == 2 || bits == 3 || bits == 4, "bits must be 2, 3 or 4 (got %d)", bits);
    SS_REQUIRE(!(bits == 2 && head_dim % 16) && !(bits == 4 && head_dim % 8),
               "head_dim %d cannot be packed at %d bits", head_dim, bits);
    SS_REQUIRE(((uintptr_t)packed % 4) == 0 && ((uintptr_t)norms % 4) == 0,
               "packed/norms must be 4-byte aligned");
    auto main = [&](const DecodeCommon &c, const DecodeShape &s, hipStream_t st) -> int {
#define SS_TURBO(DD, BB)                                                    \
    {                                                                       \
        typename VTurbo<DD, BB>::Args va{packed, norms, {},                 \
                                         static_cast<const __half *>(k_heavy), \
                                         heavy_dims, k_heavy ? n_heavy_dims : 0}; \
        for (int i = 0; i < (1 << BB); ++i) va.lv[i] = levels[i];           \
        return launch_r<DD, VTurbo<DD, BB>>(c, va, s, st, false);           \
    }
        if (head_dim == 128) {
            if (bits == 2) SS_TURBO(128, 2)
            if (bits == 3) SS_TURBO(128, 3)
            SS_TURBO(128, 4)
        }
        if (bits == 2) SS_TURBO(64, 2)
        if (bits == 3) SS_TURBO(64, 3)
        SS_TURBO(64, 4)
#undef SS_TURBO
    };
    return transformed_decode(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                              centroids, n_centroids, idx, cap, t_kv, rotation, k_buf, v_buf,
                              buf_dtype, buf_sb, buf_sh, buf_st, t_buf, causal, q_offset, out,
                              out_dtype, workspace, workspace_bytes, n_splits, stream, main,
                              kKindValu, mask);
}

extern "C" int ss_decode_attn_turboquant(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const float *norms,
    const float *levels, const float *rotation, int bits, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, void *stream) {
    return decode_attn_turboquant_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                       scale, perm, centroids, n_blocks, n_centroids, idx, packed,
                                       norms, levels, rotation, bits, cap, t_kv, k_buf, v_buf,
                                       buf_dtype, buf_sb, buf_sh, buf_st, t_buf, k_heavy,
                                       heavy_dims, n_heavy_dims, causal, q_offset, out, out_dtype,
                                       workspace, workspace_bytes, n_splits, nullptr, stream);
}

extern "C" int ss_decode_attn_turboquant_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const float *norms,
    const float *levels, const float *rotation, int bits, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    return decode_attn_turboquant_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                       scale, perm, centroids, n_blocks, n_centroids, idx, packed,
                                       norms, levels, rotation, bits, cap, t_kv, k_buf, v_buf,
                                       buf_dtype, buf_sb, buf_sh, buf_st, t_buf, k_heavy,
                                       heavy_dims, n_heavy_dims, causal, q_offset, out, out_dtype,
                                       workspace, workspace_bytes, n_splits, mask, stream);
}

static int decode_attn_grouped_hybrid_impl(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const void *scales,
    const void *zeros, int sz_dtype, int bits, int group_size, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, int causal, int64_t q_offset, void *out, int out_dtype,
    void *workspace, size_t workspace_bytes, int n_splits, const ss_attn_mask *mask, void *stream) {
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, centroids,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    if ((rc = grouped_checks(head_dim, packed, scales, zeros, sz_dtype, bits, group_size)))
        return rc;
    auto main = [&](const DecodeCommon &c, const DecodeShape &s, hipStream_t st) -> int {
        return launch_grouped(c, s, st, head_dim, packed, scales, zeros, sz_dtype, bits,
                              group_size, false);
    };
    return transformed_decode(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                              centroids, n_centroids, idx, cap, t_kv, nullptr, k_buf, v_buf,
                              buf_dtype, buf_sb, buf_sh, buf_st, t_buf, causal, q_offset, out,
                              out_dtype, workspace, workspace_bytes, n_splits, stream, main,
                              kKindValu, mask);
}

extern "C" int ss_decode_attn_grouped_hybrid(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const void *scales,
    const void *zeros, int sz_dtype, int bits, int group_size, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, int causal, int64_t q_offset, void *out, int out_dtype,
    void *workspace, size_t workspace_bytes, int n_splits, void *stream) {
    return decode_attn_grouped_hybrid_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                           scale, perm, centroids, n_blocks, n_centroids, idx,
                                           packed, scales, zeros, sz_dtype, bits, group_size, cap,
                                           t_kv, k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st,
                                           t_buf, causal, q_offset, out, out_dtype, workspace,
                                           workspace_bytes, n_splits, nullptr, stream);
}

extern "C" int ss_decode_attn_grouped_hybrid_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const void *scales,
    const void *zeros, int sz_dtype, int bits, int group_size, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, int causal, int64_t q_offset, void *out, int out_dtype,
    void *workspace, size_t workspace_bytes, int n_splits, const ss_attn_mask *mask, void *stream) {
    return decode_attn_grouped_hybrid_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                           scale, perm, centroids, n_blocks, n_centroids, idx,
                                           packed, scales, zeros, sz_dtype, bits, group_size, cap,
                                           t_kv, k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st,
                                           t_buf, causal, q_offset, out, out_dtype, workspace,
                                           workspace_bytes, n_splits, mask, stream);
}

static int decode_attn_dense_hybrid_impl(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values, int v_dtype, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, int causal, int64_t q_offset, void *out, int out_dtype,
    void *workspace, size_t workspace_bytes, int n_splits, const ss_attn_mask *mask, void *stream) {
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, centroids,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    if ((rc = dense_checks(values, v_dtype))) return rc;
    auto main = [&](const DecodeCommon &c, const DecodeShape &s, hipStream_t st) -> int {
        return launch_dense(c, s, st, head_dim, values, v_dtype, false);
    };
    return transformed_decode(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                              centroids, n_centroids, idx, cap, t_kv, nullptr, k_buf, v_buf,
                              buf_dtype, buf_sb, buf_sh, buf_st, t_buf, causal, q_offset, out,
                              out_dtype, workspace, workspace_bytes, n_splits, stream, main,
                              kKindValu, mask);
}

extern "C" int ss_decode_attn_dense_hybrid(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values, int v_dtype, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, int causal, int64_t q_offset, void *out, int out_dtype,
    void *workspace, size_t workspace_bytes, int n_splits, void *stream) {
    return decode_attn_dense_hybrid_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                         scale, perm, centroids, n_blocks, n_centroids, idx, values,
                                         v_dtype, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb,
                                         buf_sh, buf_st, t_buf, causal, q_offset, out, out_dtype,
                                         workspace, workspace_bytes, n_splits, nullptr, stream);
}

extern "C" int ss_decode_attn_dense_hybrid_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const void *values, int v_dtype, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, int causal, int64_t q_offset, void *out, int out_dtype,
    void *workspace, size_t workspace_bytes, int n_splits, const ss_attn_mask *mask, void *stream) {
    return decode_attn_dense_hybrid_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                         scale, perm, centroids, n_blocks, n_centroids, idx, values,
                                         v_dtype, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb,
                                         buf_sh, buf_st, t_buf, causal, q_offset, out, out_dtype,
                                         workspace, workspace_bytes, n_splits, mask, stream);
}

static int decode_attn_sunshape_v_impl(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint8_t *v_idx, const float *v_centroids,
    int v_block_dim, int v_n_centroids, const float *v_transform, const void *k_heavy,
    const int32_t *heavy_dims, int n_heavy_dims, int64_t cap, int64_t t_kv, const void *k_buf,
    const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, centroids,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    SS_REQUIRE(v_idx && v_centroids, "null value indices/centroids");
    SS_UNSUPPORTED(v_block_dim == 4 || v_block_dim == 8, "value block_dim %d unsupported (4 or 8)",
                   v_block_dim);
    SS_UNSUPPORTED(v_n_centroids >= 1 && v_n_centroids <= 256,
                   "value n_centroids %d unsupported (1..256, uint8 indices)", v_n_centroids);
    SS_REQUIRE(((uintptr_t)v_idx % 4) == 0, "value indices must be 4-byte aligned");
    SS_REQUIRE(((uintptr_t)v_centroids % 16) == 0, "value centroids must be 16-byte aligned");
    if (k_heavy) {
        SS_REQUIRE(heavy_dims, "null heavy_dims");
        SS_UNSUPPORTED(n_heavy_dims > 0 && n_heavy_dims % 8 == 0 && n_heavy_dims <= 64,
                       "n_heavy_dims %d unsupported (a positive multiple of 8, at most 64)",
                       n_heavy_dims);
        SS_REQUIRE(((uintptr_t)k_heavy % 16) == 0, "heavy keys must be 16-byte aligned");
    }
    // the matrix-core kernel: head_dim 128, value block_dim 4, four query
    // rows per column, 0/8/16/32/64 heavy dims, 8-byte aligned value indices
    const int nh8 = k_heavy ? n_heavy_dims / 8 : 0;
    const bool sv_mfma = head_dim == 128 && v_block_dim == 4 && ((uintptr_t)v_idx % 8) == 0 &&
                         cap < (int64_t(1) << 26) &&
                         (nh8 == 0 || nh8 == 1 || nh8 == 2 || nh8 == 4 || nh8 == 8);
    auto main = [&](const DecodeCommon &c, const DecodeShape &s, hipStream_t st) -> int {
        if (sv_mfma && s.R == kMfmaRows) {
            const typename VSunV<128, 4>::Args va{v_idx, v_centroids, v_n_centroids,
                                                  static_cast<const __half *>(k_heavy),
                                                  heavy_dims, k_heavy ? n_heavy_dims : 0};
            if (c.mask_dt != kMaskNone) {
                switch (nh8) {
                    case 1: return launch_sunv_masked<1>(c, va, s, st);
                    case 2: return launch_sunv_masked<2>(c, va, s, st);
                    case 4: return launch_sunv_masked<4>(c, va, s, st);
                    case 8: return launch_sunv_masked<8>(c, va, s, st);
                    default: return launch_sunv_masked<0>(c, va, s, st);
                }
            }
            switch (nh8) {
                case 1: return launch_sunv_mfma<1>(c, va, s, st);
                case 2: return launch_sunv_mfma<2>(c, va, s, st);
                case 4: return launch_sunv_mfma<4>(c, va, s, st);
                case 8: return launch_sunv_mfma<8>(c, va, s, st);
                default: return launch_sunv_mfma<0>(c, va, s, st);
            }
        }
#define SS_SUNV(DD, BB)                                                     \
    {                                                                       \
        typename VSunV<DD, BB>::Args va{v_idx, v_centroids, v_n_centroids,    \
                                        static_cast<const __half *>(k_heavy), \
                                        heavy_dims, k_heavy ? n_heavy_dims : 0}; \
        return launch_r<DD, VSunV<DD, BB>>(c, va, s, st, false);            \
    }
        if (head_dim == 128) {
            if (v_block_dim == 4) SS_SUNV(128, 4)
            SS_SUNV(128, 8)
        }
        if (v_block_dim == 4) SS_SUNV(64, 4)
        SS_SUNV(64, 8)
#undef SS_SUNV
    };
    // the matrix-core kernel's split policy asks no more splits (and so no
    // more workspace) than the VALU one ss_decode_turboquant_workspace_bytes
    // sizes for
    return transformed_decode(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                              centroids, n_centroids, idx, cap, t_kv, v_transform, k_buf, v_buf,
                              buf_dtype, buf_sb, buf_sh, buf_st, t_buf, causal, q_offset, out,
                              out_dtype, workspace, workspace_bytes, n_splits, stream, main,
                              sv_mfma ? kKindSunv : kKindValu, mask);
}

extern "C" int ss_decode_attn_sunshape_v(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint8_t *v_idx, const float *v_centroids,
    int v_block_dim, int v_n_centroids, const float *v_transform, const void *k_heavy,
    const int32_t *heavy_dims, int n_heavy_dims, int64_t cap, int64_t t_kv, const void *k_buf,
    const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, void *stream) {
    return decode_attn_sunshape_v_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                       scale, perm, centroids, n_blocks, n_centroids, idx, v_idx,
                                       v_centroids, v_block_dim, v_n_centroids, v_transform,
                                       k_heavy, heavy_dims, n_heavy_dims, cap, t_kv, k_buf, v_buf,
                                       buf_dtype, buf_sb, buf_sh, buf_st, t_buf, causal, q_offset,
                                       out, out_dtype, workspace, workspace_bytes, n_splits,
                                       nullptr, stream);
}

extern "C" int ss_decode_attn_sunshape_v_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const float *centroids, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint8_t *v_idx, const float *v_centroids,
    int v_block_dim, int v_n_centroids, const float *v_transform, const void *k_heavy,
    const int32_t *heavy_dims, int n_heavy_dims, int64_t cap, int64_t t_kv, const void *k_buf,
    const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    return decode_attn_sunshape_v_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                       scale, perm, centroids, n_blocks, n_centroids, idx, v_idx,
                                       v_centroids, v_block_dim, v_n_centroids, v_transform,
                                       k_heavy, heavy_dims, n_heavy_dims, cap, t_kv, k_buf, v_buf,
                                       buf_dtype, buf_sb, buf_sh, buf_st, t_buf, causal, q_offset,
                                       out, out_dtype, workspace, workspace_bytes, n_splits, mask,
                                       stream);
}
