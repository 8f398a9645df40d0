// Fused decode over token-interleaved grouped and TurboQuant codes.
#include "decode_host.hpp"

using namespace ss;

static int grouped_il_impl(const void *q, int q_dtype, int64_t batch, int n_q_heads,
                           int n_kv_heads, int64_t t_q, int head_dim, float scale,
                           const int32_t *perm, const void *codebook, int n_blocks,
                           int n_centroids, const uint8_t *idx, const uint32_t *codes_il,
                           const void *scales, const void *zeros, int sz_dtype, int bits,
                           int group_size, int64_t cap, int64_t t_kv, int causal,
                           int64_t q_offset, void *out, int out_dtype, void *workspace,
                           size_t workspace_bytes, int n_splits, const void *k_buf,
                           const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
                           int64_t buf_st, int64_t t_buf, void *stream,
                           const void *k_heavy = nullptr, const int32_t *heavy_dims = nullptr,
                           int n_heavy_dims = 0,
                           const ss_attn_mask *mask = nullptr) {
    const float *cents = static_cast<const float *>(codebook);
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, cents,
                          n_blocks, n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    SS_REQUIRE(codes_il && scales && zeros, "null codes/scales/zeros");
    SS_UNSUPPORTED(bits == 2 || bits == 4, "interleaved grouped values need bits 2 or 4 (got %d)",
                   bits);
    SS_UNSUPPORTED(group_size == head_dim || 2 * group_size == head_dim,
                   "group_size %d: the fused kernel takes one or two groups per row", group_size);
    SS_REQUIRE(sz_dtype == SS_F32 || sz_dtype == SS_F16, "scale/zero dtype must be f32 or f16");
    SS_REQUIRE(cap % 16 == 0, "cap must be a multiple of 16 for interleaved grouped values");
    SS_REQUIRE(((uintptr_t)codes_il % 16) == 0 && ((uintptr_t)scales % 16) == 0 &&
                   ((uintptr_t)zeros % 16) == 0,
               "codes, scales and zeros must be 16-byte aligned");
    SS_REQUIRE(((uintptr_t)codebook % 16) == 0, "prepared codebook must be 16-byte aligned");
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
    const int ng = head_dim / group_size;
#define SS_GIL(DD, BB, NGG, SZT)                                                              \
    {                                                                                         \
        using VF = VGil<DD, BB, NGG, SZT>;                                                    \
        SS_UNSUPPORTED(c.nhd == 0 || VF::kHeavyCapable,                                       \
                       "fp16 heavy key dims with %d-bit values at head_dim %d", BB, DD);       \
        return launch_mfma<DD, VF>(                                                           \
            c,                                                                                \
            typename VF::Args{codes_il, static_cast<const SZT *>(scales),                     \
                              static_cast<const SZT *>(zeros), k_buf, v_buf, buf_dtype,       \
                              buf_sb, buf_sh, buf_st, t_buf > 0 ? t_buf : 0},                 \
            s, st);                                                                           \
    }
#define SS_GIL_SZ(DD, BB, NGG)                     \
    {                                              \
        if (sz_dtype == SS_F16) SS_GIL(DD, BB, NGG, __half) \
        SS_GIL(DD, BB, NGG, float)                 \
    }
#define SS_GIL_NG(DD, BB)                      \
    {                                          \
        if (ng == 2) SS_GIL_SZ(DD, BB, 2)      \
        SS_GIL_SZ(DD, BB, 1)                   \
    }
    if (head_dim == 128) {
        if (bits == 2) SS_GIL_NG(128, 2)
        SS_GIL_NG(128, 4)
    }
    if (bits == 2) SS_GIL_NG(64, 2)
    SS_GIL_NG(64, 4)
#undef SS_GIL_NG
#undef SS_GIL_SZ
#undef SS_GIL
}

extern "C" int ss_decode_attn_grouped_il(const void *q, int q_dtype, int64_t batch, int n_q_heads,
                                         int n_kv_heads, int64_t t_q, int head_dim, float scale,
                                         const int32_t *perm, const void *codebook, int n_blocks,
                                         int n_centroids, const uint8_t *idx,
                                         const uint32_t *codes_il, const void *scales,
                                         const void *zeros, int sz_dtype, int bits,
                                         int group_size, int64_t cap, int64_t t_kv, int causal,
                                         int64_t q_offset, void *out, int out_dtype,
                                         void *workspace, size_t workspace_bytes, int n_splits,
                                         void *stream) {
    return grouped_il_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                           codebook, n_blocks, n_centroids, idx, codes_il, scales, zeros, sz_dtype,
                           bits, group_size, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                           workspace_bytes, n_splits, nullptr, nullptr, SS_F16, 0, 0, 0, 0, stream);
}

extern "C" int ss_decode_attn_grouped_il_hybrid(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *codes_il, const void *scales,
    const void *zeros, int sz_dtype, int bits, int group_size, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims,
    int n_heavy_dims, int causal, int64_t q_offset, void *out, int out_dtype, void *workspace,
    size_t workspace_bytes, int n_splits, void *stream) {
    SS_REQUIRE(t_buf >= 0, "negative buffer length");
    return grouped_il_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                           codebook, n_blocks, n_centroids, idx, codes_il, scales, zeros, sz_dtype,
                           bits, group_size, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                           workspace_bytes, n_splits, k_buf, v_buf, buf_dtype, buf_sb, buf_sh,
                           buf_st, t_buf, stream, k_heavy, heavy_dims, n_heavy_dims);
}

extern "C" int ss_decode_attn_grouped_il_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *codes_il, const void *scales,
    const void *zeros, int sz_dtype, int bits, int group_size, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims,
    int n_heavy_dims, int causal, int64_t q_offset, void *out, int out_dtype, void *workspace,
    size_t workspace_bytes, int n_splits, const ss_attn_mask *mask, void *stream) {
    SS_REQUIRE(t_buf >= 0, "negative buffer length");
    return grouped_il_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm,
                           codebook, n_blocks, n_centroids, idx, codes_il, scales, zeros, sz_dtype,
                           bits, group_size, cap, t_kv, causal, q_offset, out, out_dtype, workspace,
                           workspace_bytes, n_splits, k_buf, v_buf, buf_dtype, buf_sb, buf_sh,
                           buf_st, t_buf, stream, k_heavy, heavy_dims, n_heavy_dims, mask);
}

// TurboQuant values on the matrix cores (VF128 / VF64 and their arguments by
// head_dim): the checked arguments of ss_decode_attn_turboquant_il / _mfma.
template <class VF128, class VF64>
static int turboquant_mfma_decode(
    const typename VF128::Args &va128, const typename VF64::Args &va64, const void *q, int q_dtype,
    int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q, int head_dim, float scale,
    const int32_t *perm, const void *codebook, int n_blocks, int n_centroids, const uint8_t *idx,
    const float *rotation, int64_t cap, int64_t t_kv, const void *k_buf, const void *v_buf,
    int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims, int causal, int64_t q_offset,
    void *out, int out_dtype, void *workspace, size_t workspace_bytes, int n_splits,
    const ss_attn_mask *mask, void *stream) {
    const float *cents = static_cast<const float *>(codebook);
    // fused: the kernel writes out itself, rotated (one split, or its
    // in-kernel merge); else split partials for transformed_decode's merge,
    // which attends the buffered tokens, adds them and rotates
    auto launch_tq = [&](const DecodeCommon &c0, const DecodeShape &s, hipStream_t st,
                         bool fused) -> int {
        DecodeCommon c = c0;
        c.centroids = nullptr;
        c.codebook = static_cast<const uint4 *>(codebook);
        c.codebook_mul = reinterpret_cast<const float *>(
            static_cast<const char *>(codebook) + (size_t)cb_tiles(n_blocks, n_centroids) * 2 * kWave * 16);
        if (fused)
            c.rot = rotation;
        else
            c.fused_merge = 0;
        const int hrc = set_heavy(c, k_heavy, heavy_dims, n_heavy_dims);
        if (hrc) return hrc;
        if (c.mask_dt != kMaskNone) {
            SS_UNSUPPORTED(c.nhd == 0, "a mask and fp16 heavy key dims are not taken together here");
            if (head_dim == 128) return launch_mfma_masked<128, VF128>(c, va128, s, st, false);
            return launch_mfma_masked<64, VF64>(c, va64, s, st, false);
        }
        if (head_dim == 128)
            return c.nhd > 0 ? launch_mfma_kernel<128, WithHeavy<VF128>>(c, va128, s, st, false)
                             : launch_mfma_kernel<128, VF128>(c, va128, s, st, false);
        return c.nhd > 0 ? launch_mfma_kernel<64, WithHeavy<VF64>>(c, va64, s, st, false)
                         : launch_mfma_kernel<64, VF64>(c, va64, s, st, false);
    };
    if (t_buf == 0) {
        // no buffered tokens: one launch, rotation applied by the kernel
        const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits, kKindMfma);
        DecodeCommon c;
        int rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, cents, n_centroids,
                         idx, cap, t_kv, causal, q_offset, out, out_dtype, workspace, workspace_bytes,
                         head_dim);
        if (rc) return rc;
        SS_REQUIRE(((uintptr_t)rotation % 4) == 0, "misaligned rotation matrix");
        if ((rc = set_mask(c, mask))) return rc;
        if (s.S == 1 || c.fused_merge)
            return launch_tq(c, s, reinterpret_cast<hipStream_t>(stream), true);
    }
    auto main = [&](const DecodeCommon &c0, const DecodeShape &s, hipStream_t st) -> int {
        return launch_tq(c0, s, st, false);
    };
    return transformed_decode(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm, cents,
                              n_centroids, idx, cap, t_kv, rotation, k_buf, v_buf, buf_dtype, buf_sb, buf_sh,
                              buf_st, t_buf, causal, q_offset, out, out_dtype, workspace, workspace_bytes,
                              n_splits, stream, main, kKindMfma, mask);
}

static int decode_attn_turboquant_il_impl(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *codes_il, const float *norms,
    const float *levels, const float *rotation, int64_t cap, int64_t t_kv, const void *k_buf,
    const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims, int causal, int64_t q_offset,
    void *out, int out_dtype, void *workspace, size_t workspace_bytes, int n_splits,
    const ss_attn_mask *mask, void *stream) {
    const float *cents = static_cast<const float *>(codebook);
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, cents, n_blocks,
                          n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    SS_REQUIRE(codes_il && norms && levels && rotation, "null codes/norms/levels/rotation");
    SS_REQUIRE(cap % 16 == 0, "cap must be a multiple of 16 for interleaved 2-bit codes");
    SS_REQUIRE(((uintptr_t)codes_il % 16) == 0 && ((uintptr_t)norms % 16) == 0,
               "codes and norms must be 16-byte aligned");
    SS_REQUIRE(((uintptr_t)codebook % 16) == 0, "prepared codebook must be 16-byte aligned");
    // the levels must be affine in the two code bits (a symmetric table)
    const float lmax = fmaxf(fmaxf(fabsf(levels[0]), fabsf(levels[3])), 1e-30f);
    SS_UNSUPPORTED(fabsf(levels[3] - (levels[2] + levels[1] - levels[0])) <= 1e-6f * lmax,
                   "2-bit levels are not affine in the code bits (L3 != L2 + L1 - L0)");
    const float l0 = levels[0], l1 = levels[1] - levels[0], l2 = levels[2] - 2.f * levels[1] + levels[0];
    return turboquant_mfma_decode<VTq<128>, VTq<64>>(
        {codes_il, norms, l0, l1, l2}, {codes_il, norms, l0, l1, l2}, q, q_dtype, batch, n_q_heads,
        n_kv_heads, t_q, head_dim, scale, perm, codebook, n_blocks, n_centroids, idx, rotation, cap, t_kv,
        k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf, k_heavy, heavy_dims, n_heavy_dims, causal,
        q_offset, out, out_dtype, workspace, workspace_bytes, n_splits, mask, stream);
}

// One 3- or 4-bit format: its arguments from the host's levels.
template <int BITS>
static int turboquant_rows_decode(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const float *norms,
    const float *levels, const float *rotation, int64_t cap, int64_t t_kv, const void *k_buf,
    const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims, int causal, int64_t q_offset,
    void *out, int out_dtype, void *workspace, size_t workspace_bytes, int n_splits,
    const ss_attn_mask *mask, void *stream) {
    // levels times a power of two, the largest in [2^14, 2^15)
    float mx = 0.f;
    for (int i = 0; i < (1 << BITS); ++i) mx = fmaxf(mx, fabsf(levels[i]));
    SS_UNSUPPORTED(mx >= 1e-30f && mx <= 1e30f, "level table out of the fp16 split's range");
    int e;
    frexpf(mx, &e);
    static_assert(VTqRows<128, BITS>::reads_fit() && VTqRows<64, BITS>::reads_fit(),
                  "row reads leave the packed rows");
    typename VTqRows<128, BITS>::Args va128{packed, norms, {}, ldexpf(1.f, e - 15)};
    typename VTqRows<64, BITS>::Args va64{packed, norms, {}, va128.linv};
    for (int i = 0; i < (1 << BITS); ++i) va128.lv[i] = va64.lv[i] = ldexpf(levels[i], 15 - e);
    return turboquant_mfma_decode<VTqRows<128, BITS>, VTqRows<64, BITS>>(
        va128, va64, q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm, codebook,
        n_blocks, n_centroids, idx, rotation, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb, buf_sh, buf_st,
        t_buf, k_heavy, heavy_dims, n_heavy_dims, causal, q_offset, out, out_dtype, workspace,
        workspace_bytes, n_splits, mask, stream);
}

static int decode_attn_turboquant_mfma_impl(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const float *norms,
    const float *levels, const float *rotation, int bits, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    const float *cents = static_cast<const float *>(codebook);
    int rc = check_common(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, cents, n_blocks,
                          n_centroids, idx, cap, t_kv, out, out_dtype);
    if (rc) return rc;
    SS_REQUIRE(packed && norms && levels && rotation, "null packed/norms/levels/rotation");
    SS_UNSUPPORTED(bits == 3 || bits == 4, "bits %d unsupported here (3 or 4)", bits);
    SS_REQUIRE(((uintptr_t)packed % 4) == 0 && ((uintptr_t)norms % 4) == 0,
               "packed/norms must be 4-byte aligned");
    SS_REQUIRE(((uintptr_t)codebook % 16) == 0, "prepared codebook must be 16-byte aligned");
    const auto fn = bits == 3 ? turboquant_rows_decode<3> : turboquant_rows_decode<4>;
    return fn(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm, codebook, n_blocks,
              n_centroids, idx, packed, norms, levels, rotation, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb,
              buf_sh, buf_st, t_buf, k_heavy, heavy_dims, n_heavy_dims, causal, q_offset, out, out_dtype,
              workspace, workspace_bytes, n_splits, mask, stream);
}

extern "C" int ss_decode_attn_turboquant_mfma(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const float *norms,
    const float *levels, const float *rotation, int bits, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, void *stream) {
    return decode_attn_turboquant_mfma_impl(
        q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm, codebook, n_blocks,
        n_centroids, idx, packed, norms, levels, rotation, bits, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb,
        buf_sh, buf_st, t_buf, k_heavy, heavy_dims, n_heavy_dims, causal, q_offset, out, out_dtype,
        workspace, workspace_bytes, n_splits, nullptr, stream);
}

extern "C" int ss_decode_attn_turboquant_mfma_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *packed, const float *norms,
    const float *levels, const float *rotation, int bits, int64_t cap, int64_t t_kv,
    const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh,
    int64_t buf_st, int64_t t_buf, const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims,
    int causal, int64_t q_offset, void *out, int out_dtype, void *workspace, size_t workspace_bytes,
    int n_splits, const ss_attn_mask *mask, void *stream) {
    return decode_attn_turboquant_mfma_impl(
        q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim, scale, perm, codebook, n_blocks,
        n_centroids, idx, packed, norms, levels, rotation, bits, cap, t_kv, k_buf, v_buf, buf_dtype, buf_sb,
        buf_sh, buf_st, t_buf, k_heavy, heavy_dims, n_heavy_dims, causal, q_offset, out, out_dtype,
        workspace, workspace_bytes, n_splits, mask, stream);
}

extern "C" int ss_decode_attn_turboquant_il(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *codes_il, const float *norms,
    const float *levels, const float *rotation, int64_t cap, int64_t t_kv, const void *k_buf,
    const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims, int causal, int64_t q_offset,
    void *out, int out_dtype, void *workspace, size_t workspace_bytes, int n_splits, void *stream) {
    return decode_attn_turboquant_il_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                          scale, perm, codebook, n_blocks, n_centroids, idx,
                                          codes_il, norms, levels, rotation, cap, t_kv, k_buf,
                                          v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf, k_heavy,
                                          heavy_dims, n_heavy_dims, causal, q_offset, out,
                                          out_dtype, workspace, workspace_bytes, n_splits, nullptr,
                                          stream);
}

extern "C" int ss_decode_attn_turboquant_il_masked(
    const void *q, int q_dtype, int64_t batch, int n_q_heads, int n_kv_heads, int64_t t_q,
    int head_dim, float scale, const int32_t *perm, const void *codebook, int n_blocks,
    int n_centroids, const uint8_t *idx, const uint32_t *codes_il, const float *norms,
    const float *levels, const float *rotation, int64_t cap, int64_t t_kv, const void *k_buf,
    const void *v_buf, int buf_dtype, int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
    const void *k_heavy, const int32_t *heavy_dims, int n_heavy_dims, int causal, int64_t q_offset,
    void *out, int out_dtype, void *workspace, size_t workspace_bytes, int n_splits,
    const ss_attn_mask *mask, void *stream) {
    return decode_attn_turboquant_il_impl(q, q_dtype, batch, n_q_heads, n_kv_heads, t_q, head_dim,
                                          scale, perm, codebook, n_blocks, n_centroids, idx,
                                          codes_il, norms, levels, rotation, cap, t_kv, k_buf,
                                          v_buf, buf_dtype, buf_sb, buf_sh, buf_st, t_buf, k_heavy,
                                          heavy_dims, n_heavy_dims, causal, q_offset, out,
                                          out_dtype, workspace, workspace_bytes, n_splits, mask,
                                          stream);
}
