// Host side of the decodes: split plans, workspace layout, launches and the
// argument checks that the entry points of several files share.
#pragma once

#include "decode_kernels.hpp"

namespace ss {

struct DecodeShape {
    int R, n_rg, n_cols, S, tiles_per_split;
};

static int rows_per_group(int64_t rows_total) { return rows_total <= 1 ? 1 : 4; }

// Kernel families: the VALU kernel (any value layout/dtype, 4 waves per
// workgroup, 1 or 4 rows) and the MFMA kernel (fp16 values 8-token
// interleaved, 4 or 8 compute waves plus a loader wave, 4 rows).
// kKindSunv: the matrix-core SunShape-value decode (one 136 KB-LDS
// workgroup per compute unit, eight waves)
enum DecodeKind { kKindValu = 0, kKindMfma = 1, kKindSunv = 2 };
constexpr int kMfmaWaves = 4;  // fewest compute waves of an MFMA kernel (tiles per split)

static DecodeShape decode_shape(int64_t batch, int hq, int hkv, int64_t t_q, int64_t t_kv,
                                int n_splits, int kind = kKindValu) {
    DecodeShape s;
    const int64_t rows = (int64_t)(hq / hkv) * t_q;
    s.R = kind == kKindMfma ? kMfmaRows : rows_per_group(rows);
    s.n_rg = (int)((rows + s.R - 1) / s.R);
    s.n_cols = (int)(batch * hkv * s.n_rg);
    const int64_t tiles = (t_kv + kWave - 1) / kWave;
    const int waves = kind == kKindMfma ? kMfmaWaves : kind == kKindSunv ? 8 : kDecodeWaves;
    int S = n_splits;
    if (S <= 0) {
        // about one (MFMA) or two (VALU) workgroups per compute unit, each
        // with at least one 64-token tile per wave
        const int64_t target = (kind == kKindValu ? 2LL : 1LL) * device_cu_count();
        int64_t want = (target + s.n_cols - 1) / s.n_cols;
        const int64_t cap = tiles / waves;
        if (want > cap) want = cap;
        S = (int)(want < 1 ? 1 : want);
    }
    if (tiles == 0) S = 1;
    if (S > tiles && tiles > 0) S = (int)tiles;
    if (S > kMaxSplits) S = kMaxSplits;
    s.tiles_per_split = tiles > 0 ? (int)((tiles + S - 1) / S) : 0;
    if (s.tiles_per_split > 0) S = (int)((tiles + s.tiles_per_split - 1) / s.tiles_per_split);
    s.S = S;
    return s;
}

// Workspace layout: [part_cnt: kCntBytes, one int per column, spread out]
//                   [part_ml: n_cols*S*R float2, padded to 256 B]
//                   [part_acc: n_cols*S*R*D float]
// The MFMA path counts finished splits per column in part_cnt and its last
// split resets the count.  The counter area has the same place and size for
// every shape, so it must be zero before the first call on a workspace and
// then stays zero between calls; shapes with more than kCntBytes/4 columns
// merge with a separate launch instead.
constexpr size_t kCntBytes = 64 * 1024;
struct WsLayout {
    size_t cnt, ml, acc, total;
};

static WsLayout ws_layout(const DecodeShape &s, int head_dim) {
    auto pad = [](size_t b) { return (b + 255) / 256 * 256; };
    WsLayout w;
    const size_t slots = (size_t)s.n_cols * s.S * s.R;
    w.cnt = 0;
    w.ml = kCntBytes;
    w.acc = w.ml + pad(slots * 2 * sizeof(float));
    w.total = w.acc + slots * head_dim * sizeof(float);
    return w;
}

static size_t decode_ws_bytes(const DecodeShape &s, int head_dim) {
    return s.S <= 1 ? 0 : ws_layout(s, head_dim).total;
}

template <int D>
static int launch_merge(const DecodeCommon &c, const DecodeShape &s, hipStream_t st,
                        const float *rot = nullptr, void *rot_out = nullptr, int rot_dtype = 0,
                        const MergeBuffer &mb = MergeBuffer{}) {
    if (s.S <= 1) return SS_OK;
    auto merge = mb.n > 0 ? decode_merge_kernel<D, true> : decode_merge_kernel<D, false>;
    hipLaunchKernelGGL(merge, dim3(s.n_cols, s.R), dim3(kDecodeThreads), 0, st, c, s.R, rot,
                       rot_out, rot_dtype, mb);
    SS_LAUNCH_CHECK("decode_merge_kernel launch");
    return SS_OK;
}

// Once per instance of the matrix-core decode kernel: the device must hold
// its LDS, and its dynamic LDS size is set.
template <int D, class VF>
static int mfma_kernel_setup() {
    constexpr int NC = VF::kComputeWaves;
    using K = WsCfg<D, NC, VF>;
    auto kern = decode_attn_mfma_kernel<D, NC, VF>;
    static bool done = false;
    if (done) return SS_OK;
    int dev = 0, max_lds = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&max_lds, hipDeviceAttributeSharedMemPerBlockOptin, dev);
    if (e != hipSuccess) return hip_fail(e, "hipDeviceGetAttribute(LDS)");
    SS_UNSUPPORTED(max_lds >= K::kLds, "decode needs %d bytes of LDS per workgroup, device has %d", K::kLds,
                   max_lds);
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            K::kLds);
    if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(decode mfma)");
    done = true;
    return SS_OK;
}

template <int D, class VF>
static int launch_mfma_kernel(DecodeCommon c, const typename VF::Args &va, const DecodeShape &s,
                              hipStream_t st, bool merge = true) {
    constexpr int NC = VF::kComputeWaves;
    using K = WsCfg<D, NC, VF>;
    auto kern = decode_attn_mfma_kernel<D, NC, VF>;
    const int rc = mfma_kernel_setup<D, VF>();
    if (rc) return rc;
    hipLaunchKernelGGL(kern, dim3(s.S, s.n_cols), dim3(K::kWaves * kWave), K::kLds, st, c, va);
    SS_LAUNCH_CHECK("decode_attn_mfma_kernel launch");
    if (c.fused_merge || !merge) return SS_OK;  // the kernel (or the caller) merges the splits
    return launch_merge<D>(c, s, st);
}

// launch_mfma_kernel<D, WithMask<VF>>, compiled in decode_masked.hip for the
// formats launch_mfma passes on
template <int D, class VF>
int launch_mfma_masked(const DecodeCommon &c, const typename VF::Args &va, const DecodeShape &s,
                       hipStream_t st, bool merge = true);

// the format's kernel, or its heavy-dim variant when the call carries fp16
// heavy key dims, or its masked one
template <int D, class VF>
static int launch_mfma(DecodeCommon c, const typename VF::Args &va, const DecodeShape &s,
                       hipStream_t st) {
    if (c.mask_dt != kMaskNone) {
        SS_UNSUPPORTED(c.nhd == 0, "a mask and fp16 heavy key dims are not taken together here");
        if constexpr (!StepShareOf<VF>::value && !std::is_same<VF, VIl8<D>>::value)
            return launch_mfma_masked<D, VF>(c, va, s, st);
        SS_UNSUPPORTED(false, "this decode shape takes no mask");
    }
    if (c.nhd > 0) {
        if constexpr (VfHeavyCapable<VF>::value)
            return launch_mfma_kernel<D, WithHeavy<VF>>(c, va, s, st);
        SS_UNSUPPORTED(false, "fp16 heavy key dims are not taken by this decode shape");
    }
    return launch_mfma_kernel<D, VF>(c, va, s, st);
}

template <int NH8, bool MK = false>
static int launch_sunv_mfma(const DecodeCommon &c, const typename VSunV<128, 4>::Args &va,
                            const DecodeShape &s, hipStream_t st) {
    auto kern = sunv_mfma_kernel<NH8, MK>;
    static bool attr_set = false;  // per instantiation
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 kSvLdsBytes);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(sunv mfma)");
        attr_set = true;
    }
    hipLaunchKernelGGL(kern, dim3(s.S, s.n_cols), dim3(kSvWaves * kWave), kSvLdsBytes, st, c, va);
    SS_LAUNCH_CHECK("sunv_mfma_kernel launch");
    return SS_OK;
}

// launch_sunv_mfma<NH8, true>, compiled in decode_masked.hip
template <int NH8>
int launch_sunv_masked(const DecodeCommon &c, const typename VSunV<128, 4>::Args &va,
                       const DecodeShape &s, hipStream_t st);

template <int D, int R, class VF, bool MK>
static int launch_mk(DecodeCommon c, const typename VF::Args &va, const DecodeShape &s,
                  hipStream_t st, bool merge = true) {
    constexpr int TH = VfThreads<VF>::value;
    const size_t lds = decode_lds_bytes<D, R, TH / kWave>() + VfLds<VF>::value;
    auto kern = decode_attn_kernel<D, R, VF, MK>;
    static bool attr_set = false;  // per instantiation
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(decode)");
        attr_set = true;
    }
    dim3 grid(s.S, s.n_cols, VfSlabs<VF>::value);
    hipLaunchKernelGGL(kern, grid, dim3(TH), lds, st, c, va);
    SS_LAUNCH_CHECK("decode_attn_kernel launch");
    return merge ? launch_merge<D>(c, s, st) : SS_OK;
}

template <int D, int R, class VF>
static int launch(DecodeCommon c, const typename VF::Args &va, const DecodeShape &s, hipStream_t st,
                  bool merge = true) {
    return c.mask_dt != kMaskNone ? launch_mk<D, R, VF, true>(c, va, s, st, merge)
                                  : launch_mk<D, R, VF, false>(c, va, s, st, merge);
}

template <int D, class VF>
static int launch_r(DecodeCommon c, const typename VF::Args &va, const DecodeShape &s,
                    hipStream_t st, bool merge = true) {
    if (s.R == 1) return launch<D, 1, VF>(c, va, s, st, merge);
    return launch<D, 4, VF>(c, va, s, st, merge);
}

static int check_common(const void *q, int q_dtype, int64_t batch, int hq, int hkv, int64_t t_q,
                        int head_dim, const float *centroids, int n_blocks, int n_centroids,
                        const uint8_t *idx, int64_t cap, int64_t t_kv, void *out, int out_dtype) {
    SS_REQUIRE(q && centroids && idx && out, "null pointer argument");
    SS_REQUIRE(valid_dtype(q_dtype) && valid_dtype(out_dtype), "bad dtype code");
    SS_REQUIRE(batch >= 1 && hq >= 1 && hkv >= 1 && t_q >= 1, "empty batch/heads/t_q");
    SS_REQUIRE(hq % hkv == 0, "n_q_heads (%d) must be a multiple of n_kv_heads (%d)", hq, hkv);
    SS_UNSUPPORTED(head_dim == 64 || head_dim == 128,
                   "head_dim %d unsupported (64 or 128)", head_dim);
    SS_UNSUPPORTED(n_blocks * kBlockDim == head_dim,
                   "fused kernel needs block_dim 8 (n_blocks %d, head_dim %d)", n_blocks, head_dim);
    SS_UNSUPPORTED(n_centroids >= 1 && n_centroids <= 256,
                   "n_centroids %d unsupported (1..256, uint8 indices)", n_centroids);
    SS_REQUIRE(t_kv >= 0 && t_kv <= cap, "t_kv %lld outside [0, cap=%lld]", (long long)t_kv,
               (long long)cap);
    SS_REQUIRE(((uintptr_t)idx % 16) == 0, "idx must be 16-byte aligned");
    SS_REQUIRE(((uintptr_t)centroids % 16) == 0, "centroids must be 16-byte aligned");
    return SS_OK;
}

// A call's attention mask (null or data null: none).
static int set_mask(DecodeCommon &c, const ss_attn_mask *mask) {
    if (!mask || !mask->data) return SS_OK;
    SS_REQUIRE(mask->type >= SS_MASK_BOOL && mask->type <= SS_MASK_F32, "bad mask type %d", mask->type);
    SS_REQUIRE(mask->sb >= 0 && mask->sh >= 0 && mask->sq >= 0, "negative mask strides");
    static_assert((int)kMaskBool == SS_MASK_BOOL && (int)kMaskF16 == SS_MASK_F16 &&
                      (int)kMaskBf16 == SS_MASK_BF16 && (int)kMaskF32 == SS_MASK_F32, "mask types");
    const int es = mask->type == SS_MASK_BOOL ? 1 : mask->type == SS_MASK_F32 ? 4 : 2;
    SS_REQUIRE((uintptr_t)mask->data % es == 0, "mask not aligned to its elements");
    SS_REQUIRE(!c.causal, "an array mask replaces the causal one");
    c.mask = mask->data;
    c.mask_dt = mask->type;
    c.m_sb = mask->sb;
    c.m_sh = mask->sh;
    c.m_sq = mask->sq;
    return SS_OK;
}

// The arguments of a decode launch (decode.hip); checks the workspace.
int fill_common(DecodeCommon &c, const DecodeShape &s, const void *q, int q_dtype,
                int hq, int hkv, int64_t t_q, float scale, const int32_t *perm,
                const float *centroids, int n_centroids, const uint8_t *idx, int64_t cap,
                int64_t t_kv, int causal, int64_t q_offset, void *out, int out_dtype,
                void *ws, size_t ws_bytes, int head_dim);

static int dense_checks(const void *values, int v_dtype) {
    SS_REQUIRE(values, "null values");
    SS_REQUIRE(valid_dtype(v_dtype), "bad value dtype");
    SS_REQUIRE(((uintptr_t)values % 16) == 0, "values must be 16-byte aligned");
    return SS_OK;
}

static int grouped_checks(int head_dim, const uint32_t *packed, const void *scales,
                          const void *zeros, int sz_dtype, int bits, int group_size) {
    SS_REQUIRE(packed && scales && zeros, "null packed/scales/zeros");
    SS_REQUIRE(bits == 2 || bits == 3 || bits == 4, "bits must be 2, 3 or 4 (got %d)", bits);
    SS_REQUIRE(sz_dtype == SS_F32 || sz_dtype == SS_F16, "scale/zero dtype must be f32 or f16");
    SS_REQUIRE(group_size >= 1 && head_dim % group_size == 0,
               "head_dim %d not divisible by group_size %d", head_dim, group_size);
    SS_REQUIRE(!(bits == 2 && head_dim % 16) && !(bits == 4 && head_dim % 8),
               "head_dim %d cannot be packed at %d bits", head_dim, bits);
    // a packed word spans at most two scale groups
    SS_UNSUPPORTED(group_size >= 32 / bits, "group_size %d < %d values per word", group_size,
                   32 / bits);
    SS_REQUIRE(((uintptr_t)packed % 4) == 0, "packed values must be 4-byte aligned");
    return SS_OK;
}

// Workspace of the TurboQuant decode: the split partials (as for the other
// VALU decodes), then the fp32 output rows of the rotated basis.  A buffer
// adds a slot per column: nothing is stored there, it makes a single split
// write its partial for the merge, which attends the buffered tokens itself.
static DecodeShape with_buffer_slot(DecodeShape s, int64_t t_buf) {
    if (t_buf > 0) s.S += 1;
    return s;
}

static size_t turboquant_ws_bytes(const DecodeShape &sw, int64_t rows, int head_dim) {
    // the rows never overlap the split counters at the workspace's start,
    // which the matrix-core decodes sharing this workspace rely on being zero
    // (with one split there are no partials, but the counter area stays)
    size_t part = decode_ws_bytes(sw, head_dim);
    if (part < kCntBytes) part = kCntBytes;
    part = (part + 255) / 256 * 256;
    return part + (size_t)rows * head_dim * sizeof(float);
}

// Shared host side of the decodes whose values accumulate in a transformed
// basis (TurboQuant's rotation, a SunShape value codec's permutation or
// rotation): the VALU decode writes y (fp32, that basis) or split partials;
// the merge launch attends buffered original-basis tokens and adds them after
// the transform; it, or rotate_rows_kernel for a single split without a
// buffer, writes out = y @ transform in out_dtype.  A null
// transform is the identity (values in the original basis: the grouped and
// dense VALU decodes with a hybrid cache's buffer): the kernels and the merge
// write out directly.
template <class MainLaunch>
static int transformed_decode(const void *q, int q_dtype, int64_t batch, int hq, int hkv,
                              int64_t t_q, int head_dim, float scale, const int32_t *perm,
                              const float *centroids, int n_centroids, const uint8_t *idx,
                              int64_t cap, int64_t t_kv, const float *transform,
                              const void *k_buf, const void *v_buf, int buf_dtype,
                              int64_t buf_sb, int64_t buf_sh, int64_t buf_st, int64_t t_buf,
                              int causal, int64_t q_offset, void *out, int out_dtype,
                              void *workspace, size_t workspace_bytes, int n_splits,
                              void *stream, MainLaunch &&launch_main, int kind = kKindValu,
                              const ss_attn_mask *mask = nullptr) {
    const bool ident = transform == nullptr;
    SS_REQUIRE(((uintptr_t)transform % 4) == 0, "misaligned transform/rotation matrix");
    SS_REQUIRE(t_buf >= 0, "negative buffer length");
    if (t_buf > 0) {
        SS_REQUIRE(k_buf && v_buf, "null buffer keys/values");
        SS_REQUIRE(buf_dtype == SS_F16 || buf_dtype == SS_BF16 || buf_dtype == SS_F32,
                   "buffer dtype must be f16, bf16 or f32");
        SS_REQUIRE(buf_sb >= 0 && buf_sh >= 0 && buf_st >= head_dim,
                   "buffer strides must be non-negative, token stride >= head_dim");
    }
    const DecodeShape s = decode_shape(batch, hq, hkv, t_q, t_kv, n_splits, kind);
    const DecodeShape sw = with_buffer_slot(s, t_buf);  // partial slots incl. the buffer's
    const int64_t rows = batch * hq * t_q;
    const size_t need = turboquant_ws_bytes(sw, rows, head_dim);
    if (!workspace || workspace_bytes < need) {
        set_error("decode workspace too small: need %zu bytes, got %zu", need,
                  workspace ? workspace_bytes : (size_t)0);
        return SS_ERR_WORKSPACE;
    }
    SS_REQUIRE(((uintptr_t)workspace % 256) == 0, "workspace must be 256-byte aligned");
    float *y = reinterpret_cast<float *>(static_cast<char *>(workspace) + need -
                                         (size_t)rows * head_dim * sizeof(float));
    DecodeCommon c;
    int rc = fill_common(c, sw, q, q_dtype, hq, hkv, t_q, scale, perm, centroids, n_centroids,
                         idx, cap, t_kv, causal, q_offset, ident ? out : y,
                         ident ? out_dtype : SS_F32, workspace, workspace_bytes, head_dim);
    if (rc) return rc;
    if ((rc = set_mask(c, mask))) return rc;
    c.tiles_per_split = s.tiles_per_split;  // the compressed tokens' splits: grid s.S
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    rc = launch_main(c, s, st);  // no merge: it follows, with the buffer
    if (rc) return rc;
    MergeBuffer mb{};
    if (t_buf > 0) {
        const int64_t es = buf_dtype == SS_F32 ? 4 : 2;
        const bool vec = (((uintptr_t)k_buf | (uintptr_t)v_buf) % 16) == 0 &&
                         ((buf_sb | buf_sh | buf_st) * es) % 16 == 0;
        mb = MergeBuffer{k_buf, v_buf, buf_dtype, vec ? 1 : 0, buf_sb, buf_sh, buf_st, t_buf};
    }
    if (sw.S > 1)
        return head_dim == 128 ? launch_merge<128>(c, sw, st, transform, out, out_dtype, mb)
                               : launch_merge<64>(c, sw, st, transform, out, out_dtype, mb);
    if (ident) return SS_OK;  // the one split wrote out
    const unsigned blocks = (unsigned)((rows + kRotRows - 1) / kRotRows);
    if (head_dim == 128)
        hipLaunchKernelGGL(rotate_rows_kernel<128>, dim3(blocks), dim3(256), 0, st, y, transform,
                           rows, out, out_dtype);
    else
        hipLaunchKernelGGL(rotate_rows_kernel<64>, dim3(blocks), dim3(256), 0, st, y, transform,
                           rows, out, out_dtype);
    SS_LAUNCH_CHECK("rotate_rows_kernel launch");
    return SS_OK;
}

// Tiles of the prepared codebook: 16 centroids of 4 consecutive blocks.
__host__ __device__ inline int cb_tiles(int n_blocks, int n_centroids) {
    return (n_blocks / 4) * ((n_centroids + 15) / 16);
}

// Checks shared by the hybrid entry points: t_buf buffered tokens at k_buf /
// v_buf with element strides buf_sb, buf_sh, buf_st.
static int check_buffer(const void *k_buf, const void *v_buf, int buf_dtype, int64_t buf_sb,
                        int64_t buf_sh, int64_t buf_st, int64_t t_buf, int head_dim) {
    SS_REQUIRE(t_buf >= 0, "negative buffer length");
    if (t_buf == 0) return SS_OK;
    SS_REQUIRE(k_buf && v_buf, "null buffer keys/values");
    SS_REQUIRE(buf_dtype == SS_F16 || buf_dtype == SS_BF16 || buf_dtype == SS_F32,
               "buffer dtype must be f16, bf16 or f32");
    SS_REQUIRE(buf_sb >= 0 && buf_sh >= 0 && buf_st >= head_dim,
               "buffer strides must be non-negative, token stride >= head_dim");
    SS_REQUIRE(((uintptr_t)k_buf % 16) == 0 && buf_sb % 8 == 0 && buf_sh % 8 == 0 &&
                   buf_st % 8 == 0,
               "buffer keys must be 16-byte aligned with strides a multiple of 8 elements");
    return SS_OK;
}

// fp16 heavy-block key dims of a mixed-precision codec for the matrix-core
// kernels (hybrid caches): [rows][n] halves at 16-byte aligned rows.
static int set_heavy(DecodeCommon &c, const void *k_heavy, const int32_t *heavy_dims, int n) {
    if (!k_heavy) return SS_OK;
    SS_REQUIRE(heavy_dims, "null heavy_dims");
    SS_UNSUPPORTED(n > 0 && n % 8 == 0 && n <= kMaxHeavyMfma,
                   "n_heavy_dims %d unsupported (a positive multiple of 8, at most %d)", n,
                   kMaxHeavyMfma);
    SS_REQUIRE(((uintptr_t)k_heavy % 16) == 0, "heavy keys must be 16-byte aligned");
    c.kheavy = static_cast<const __half *>(k_heavy);
    c.heavy_dims = heavy_dims;
    c.nhd = n;
    return SS_OK;
}

}  // namespace ss
