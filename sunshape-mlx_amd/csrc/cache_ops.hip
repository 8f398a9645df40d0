// KV-cache value layout: append tokens into the 8-token interleaved fp16 layout.
//
// The decode kernel's MFMA path reads values as [cap/8][head_dim][8] per
// (batch, KV head): the 8 consecutive tokens of one dim are 16 contiguous
// bytes, the K-major operand of v_mfma_f32_16x16x32_f16.  Appending T new
// tokens at position `offset` scatters each token's head_dim values with a
// 16-byte stride; the index cache keeps the token-major [cap][n_blocks]
// layout of the reference (cache.py:102-150).
#include "ss_common.hpp"

namespace ss {

// A thread takes two dims of one 8-token block: eight 4-byte loads (a wave's
// cover 256 consecutive bytes of each token's row) and two 16-byte stores (2
// KB a wave).  Blocks at the ends of the range that hold other tokens too
// store only their own.  HBM bounds it.  One element a thread, its 2-byte
// stores 16 bytes apart, took 17.1 us for 8 heads x 4096 tokens of 128 dims.
// OUT_BF: bfloat16 words out (the input must be bfloat16), else fp16.
template <bool OUT_BF>
__global__ void __launch_bounds__(256)
    append_il8_kernel(const void *v, int v_dtype, int64_t n_h, int64_t n_t, int64_t n_blk, int64_t total,
                      int64_t v_sb, int64_t v_sh, int64_t v_st, int d, int pairs, __half *out, int64_t cap,
                      int64_t offset) {
    const int per = pairs ? (d + 1) / 2 : d;  // threads of a block's row
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= total) return;
    const int64_t n = e / per;
    const int j = (int)(e - n * per) * (pairs ? 2 : 1);
    const int64_t bh = n / n_blk, blk = offset / 8 + (n - bh * n_blk);
    const int64_t b = bh / n_h, h = bh - b * n_h;
    const int64_t t0 = blk * 8 - offset;  // token of the block's first slot (may be < 0)
    const int64_t src = b * v_sb + h * v_sh + j;
    const bool whole = t0 >= 0 && t0 + 8 <= n_t && ((uintptr_t)out % 16) == 0;
    uint32_t w[8];  // dims j (low half) and j + 1 of the block's tokens
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t t = min(max(t0 + i, (int64_t)0), n_t - 1);
        const int64_t o = src + t * v_st;
        if (OUT_BF || v_dtype == SS_F16) {
            const uint16_t *p = static_cast<const uint16_t *>(v) + o;
            w[i] = pairs ? *reinterpret_cast<const uint32_t *>(p) : *p;
        } else {
            const __half x0 = __float2half(load_as_f32(v, v_dtype, o));
            const __half x1 = pairs ? __float2half(load_as_f32(v, v_dtype, o + 1)) : x0;
            w[i] = (uint32_t)__half_as_ushort(x0) | ((uint32_t)__half_as_ushort(x1) << 16);
        }
    }
    uint16_t *dst = reinterpret_cast<uint16_t *>(out) + ((bh * (cap / 8) + blk) * d + j) * 8;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if (k == 1 && !pairs) break;
        const int sh = 16 * k;
        if (whole) {
            uint32_t o4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                o4[i] = ((w[2 * i] >> sh) & 0xffffu) | (((w[2 * i + 1] >> sh) & 0xffffu) << 16);
            *reinterpret_cast<uint4 *>(dst + 8 * k) = make_uint4(o4[0], o4[1], o4[2], o4[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (t0 + i >= 0 && t0 + i < n_t) dst[8 * k + i] = (uint16_t)(w[i] >> sh);
        }
    }
}

// Whole keys for the hybrid prompt kernel: one wave per token.  Dim j of the
// output is dim perm[j] of the key (the codec's basis; perm null = identity).
// With s = row_exp_shift(max |key|), row 0 = fp16(key * 2^-s) and row 1 =
// fp16(key * 2^-s - row 0); factor = 2^s.  Multiplying by a power of two is
// exact, so row 0 + row 1 is the key times 2^-s to 22 significant bits, and
// exactly for fp16 and bf16 keys (row 1 = 0); a remainder below fp16's
// normal range is rounded there, under 2^-38 of the row's largest element.
__global__ void __launch_bounds__(256)
    raw_key_rows_kernel(const void *k, int k_dtype, int64_t n_h, int64_t n_t, int64_t n_tok,
                        int64_t k_sb, int64_t k_sh, int64_t k_st, int d, const int32_t *perm,
                        __half *rows, float *fac) {
    const int64_t n = (int64_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
    const int lane = threadIdx.x & 63;
    if (n >= n_tok) return;  // whole waves leave together
    const int64_t b = n / (n_h * n_t);
    const int64_t rem = n - b * n_h * n_t;
    const int64_t h = rem / n_t;
    const int64_t t = rem - h * n_t;
    const int64_t base = b * k_sb + h * k_sh + t * k_st;
    float m = 0.f;
    for (int j = lane; j < d; j += 64)
        m = fmaxf(m, fabsf(load_as_f32(k, k_dtype, base + (perm ? perm[j] : j))));
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    const int s = row_exp_shift(m);
    const float down = exp2i(-s);
    __half *r0 = rows + n * 2 * d;
    for (int j = lane; j < d; j += 64) {
        const float x = load_as_f32(k, k_dtype, base + (perm ? perm[j] : j)) * down;
        const __half hi = __float2half(x);
        r0[j] = hi;
        r0[d + j] = __float2half(x - __half2float(hi));
    }
    if (lane == 0) fac[n] = exp2i(s);
}

}  // namespace ss

using namespace ss;

template <bool OUT_BF>
static int append_il8(const void *values, int v_dtype, int64_t n_b, int64_t n_h, int64_t n_t,
                      int64_t v_sb, int64_t v_sh, int64_t v_st, int head_dim, void *out_il8,
                      int64_t cap, int64_t offset, void *stream) {
    SS_REQUIRE(valid_dtype(v_dtype), "bad value dtype");
    SS_REQUIRE(n_b >= 0 && n_h >= 0 && n_t >= 0 && head_dim >= 1, "bad sizes");
    SS_REQUIRE(cap % 8 == 0, "cap must be a multiple of 8");
    SS_REQUIRE(offset >= 0 && offset + n_t <= cap, "tokens [%lld, %lld) exceed cap %lld",
               (long long)offset, (long long)(offset + n_t), (long long)cap);
    if (n_b * n_h * n_t == 0) return SS_OK;
    SS_REQUIRE(values && out_il8, "null pointer argument");
    // two dims a thread where every row starts on a pair of elements
    const int es = v_dtype == SS_F32 ? 4 : 2;
    const bool pairs = head_dim % 2 == 0 && ((uintptr_t)values % (2 * es)) == 0 &&
                       ((v_sb | v_sh | v_st) & 1) == 0;
    const int64_t n_blk = (offset + n_t + 7) / 8 - offset / 8;
    const int64_t total = n_b * n_h * n_blk * (pairs ? head_dim / 2 : head_dim);
    SS_UNSUPPORTED(n_b * n_h * n_t * head_dim < (1LL << 32) && total < (1LL << 39),
                   "too many elements for one launch");
    hipLaunchKernelGGL(append_il8_kernel<OUT_BF>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), values, v_dtype, n_h, n_t, n_blk, total,
                       v_sb, v_sh, v_st, head_dim, pairs ? 1 : 0, reinterpret_cast<__half *>(out_il8),
                       cap, offset);
    SS_LAUNCH_CHECK("append_il8_kernel launch");
    return SS_OK;
}

extern "C" int ss_append_values_il8(const void *values, int v_dtype, int64_t n_b, int64_t n_h,
                                    int64_t n_t, int64_t v_sb, int64_t v_sh, int64_t v_st,
                                    int head_dim, void *out_il8, int64_t cap, int64_t offset,
                                    void *stream) {
    return append_il8<false>(values, v_dtype, n_b, n_h, n_t, v_sb, v_sh, v_st, head_dim, out_il8, cap,
                             offset, stream);
}

extern "C" int ss_append_values_il8_bf16(const void *values, int64_t n_b, int64_t n_h, int64_t n_t,
                                         int64_t v_sb, int64_t v_sh, int64_t v_st, int head_dim,
                                         void *out_il8, int64_t cap, int64_t offset, void *stream) {
    return append_il8<true>(values, SS_BF16, n_b, n_h, n_t, v_sb, v_sh, v_st, head_dim, out_il8, cap,
                            offset, stream);
}

extern "C" int ss_raw_key_rows(const void *keys, int k_dtype, int64_t n_b, int64_t n_h,
                               int64_t n_t, int64_t k_sb, int64_t k_sh, int64_t k_st,
                               int head_dim, const int32_t *perm, void *rows, float *factors,
                               void *stream) {
    SS_REQUIRE(valid_dtype(k_dtype), "bad key dtype");
    SS_REQUIRE(n_b >= 0 && n_h >= 0 && n_t >= 0 && head_dim >= 1, "bad sizes");
    const int64_t n_tok = n_b * n_h * n_t;
    if (n_tok == 0) return SS_OK;
    SS_REQUIRE(keys && rows && factors, "null pointer argument");
    SS_UNSUPPORTED(n_tok < (1LL << 31), "too many tokens for one launch");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(raw_key_rows_kernel, dim3((unsigned)((n_tok + 3) / 4)), dim3(256), 0, st,
                       keys, k_dtype, n_h, n_t, n_tok, k_sb, k_sh, k_st, head_dim, perm,
                       reinterpret_cast<__half *>(rows), factors);
    SS_LAUNCH_CHECK("raw_key_rows_kernel launch");
    return SS_OK;
}
