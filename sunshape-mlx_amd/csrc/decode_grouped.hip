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
    typename VTq<128>::Args va128{codes_il, norms, levels[0], levels[1] - levels[0],
                                  levels[2] - 2.f * levels[1] + levels[0]};
    // fused: the kernel writes out itself, rotated (one split, or its
    // in-kernel merge); else split partials that transformed_decode merges
    // with the buffer's partial and rotates
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
            if (head_dim == 128) return launch_mfma_masked<128, VTq<128>>(c, va128, s, st, false);
            const typename VTq<64>::Args va64{va128.codes, va128.norms, va128.l0, va128.l1, va128.l2};
            return launch_mfma_masked<64, VTq<64>>(c, va64, s, st, false);
        }
        auto go = [&](auto dd, auto vf) -> int {
            constexpr int DD = decltype(dd)::value;
            using VF = typename decltype(vf)::type;
            constexpr int NC = VF::kComputeWaves;
            using K = WsCfg<DD, NC, VF>;
            auto kern = decode_attn_mfma_kernel<DD, NC, VF>;
            const int src = mfma_kernel_setup<DD, VF>();
            if (src) return src;
            const typename VF::Args va{va128.codes, va128.norms, va128.l0, va128.l1, va128.l2};
            hipLaunchKernelGGL(kern, dim3(s.S, s.n_cols), dim3(K::kWaves * kWave), K::kLds, st, c, va);
            SS_LAUNCH_CHECK("decode_attn_mfma_kernel (turboquant) launch");
            return SS_OK;
        };
        using I128 = std::integral_constant<int, 128>;
        using I64 = std::integral_constant<int, 64>;
        if (c.nhd > 0)
            return head_dim == 128 ? go(I128{}, TypeTag<WithHeavy<VTq<128>>>{})
                                   : go(I64{}, TypeTag<WithHeavy<VTq<64>>>{});
        return head_dim == 128 ? go(I128{}, TypeTag<VTq<128>>{})
                               : go(I64{}, TypeTag<VTq<64>>{});
    };
    if (t_buf == 0) {
        // no buffered tokens: one launch, rotation applied by the kernel
        const DecodeShape s = decode_shape(batch, n_q_heads, n_kv_heads, t_q, t_kv, n_splits, kKindMfma);
        DecodeCommon c;
        rc = fill_common(c, s, q, q_dtype, n_q_heads, n_kv_heads, t_q, scale, perm, cents, n_centroids,
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
