// Prompt attention over block-VQ keys in two launches: the keys are
// reconstructed once per (batch, KV head) as matrix-core operands, then every
// workgroup streams them through LDS.
//
// prefill32_il8_kernel (prefill.hip) gathers each key row from a codebook copy
// in LDS, once per wave of 32 query rows: 16 random 16-byte reads a lane and
// sub-tile, whose bank conflicts double their cost, each waited for before its
// product.  Here prefill_keys_kernel writes the operand fragments themselves
// (512 bytes a token and KV head at head_dim 128, O(T) work), so the attention
// kernel's LDS reads are lane-contiguous and go out together.
//
// prefill_frag_kernel: S^T = Khat Q'^T and O = P V on the 32x32x16 products,
// as prefill32 (lane l holds row l%32; entries of S^T are the A operand of
// P V).  A workgroup of RW x KW waves takes 32 RW query rows (flattened
// position x head of one KV group, so any group size fits) and KW sub-tiles
// of 32 tokens at a time: wave (kg, rw) attends sub-tile kg of each tile for
// rows 32 rw ..; the KW partial softmaxes of a row meet in LDS at the end.
// Key and value tiles stream through kStages LDS stages (global_load_lds, one
// barrier a tile, the copies two or three tiles ahead), issued after the
// tile's own LDS reads.
//
// Bound: the chain product -> softmax -> product of two waves a SIMD; the
// matrix cores are busy for a third of the time (1.5 products per attention
// product, the keys' hi and lo parts), and with the products, the copies or
// the exponentials taken out the rest takes 75, 89 and 93 % of the time.
// 32/8 heads of 128 dims, prefill32 before: 4096 tokens 335 -> 258 us (533
// TFLOP/s of attention), 2 x 512 tokens after 8192 367 -> 280 us; bf16 values,
// 2041 tokens, 1146 us on the vector-ALU decode before, 119 to 127 now.
//
// Values: fp16, P as one fp16 operand of p * 2^11 (as prefill32) or as its hi
// and lo parts (22 bits, as the decode kernels; ss_prefill_attn chooses), or
// bfloat16 with P as three bfloat16 parts (24 bits, float32's own; all above
// zero, so that an infinite value stays infinite where it is seen).
#include "ss_common.hpp"

#include <algorithm>
#include <type_traits>

namespace ss {

namespace {

typedef _Float16 pg_f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 pg_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 pg_bf16x8 __attribute__((ext_vector_type(8)));
typedef float pg_f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 pg_f16x2 __attribute__((ext_vector_type(2)));
typedef float pg_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t pg_u32x2 __attribute__((ext_vector_type(2)));

template <class T>
using pg_lds = __attribute__((address_space(3))) T;

// A row keeps its running maximum while a sub-tile's scores stay within kPgLag
// log2 units above it; probabilities are staged times 2^kPgExp (fp16: below
// the fp16 maximum at 2^(kPgExp + kPgLag)).
constexpr float kPgLag = 4.f;
constexpr float kPgExp = 11.f;
constexpr float kPgMore = 1.f + 0x1p-23f;

struct FragArgs {
    const void *q;
    int q_dtype;
    int n_q_heads, n_kv_heads, rep;
    int64_t t_q;
    float scale;
    const int32_t *perm;
    const uint4 *codebook;  // prepared split-fp16 tiles (ss_codebook_f16x2)
    const float *cb_mul;    // their power-of-two multiplier
    int nct;                // centroid tiles of 16
    const uint8_t *idx;     // [B][Hkv][cap][D/8]
    const void *v8;         // [B][Hkv][cap_v/8][D][8]
    int64_t cap, cap_v, t_kv;
    // whole keys from position t_raw0 on (ss_raw_key_rows), or null
    const __half *kraw;
    const float *kfac;
    int64_t t_raw0, n_raw;
    int causal;
    int64_t q_offset;
    void *out;
    int out_dtype;
    int64_t bh0;            // first (batch, KV head) of this launch
    uint4 *frag;            // key fragments of the launch's heads
    int64_t n_sub;          // sub-tiles of a head (a multiple of KW)
    int n_rt;               // row tiles
};

__device__ __forceinline__ float pg_lane(float x, int src) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(x)));
}

// The high halves of two words as one, a's the lower.
__device__ __forceinline__ uint32_t pg_high_halves(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

template <int N>
__device__ __forceinline__ void pg_wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

}  // namespace

// Key fragments of sub-tile blockIdx.x of head bh0 + blockIdx.y: for k-step ks
// (16 dims), lane l of the A operand holds token l%32's dims 16 ks + 8 (l/32)
// .. +7, i.e. the codebook row of block 2 ks + l/32; the hi parts of the D/16
// k-steps (1 KB each), then the lo parts in the hi units (lo * 2^-11, as
// prefill32's LDS copy).  Whole keys (from t_raw0) take their two rows.  HBM
// bounds it: 16 index bytes in, 512 bytes out a token (D = 128).
template <int D>
__global__ void __launch_bounds__(256) prefill_keys_kernel(FragArgs a) {
    constexpr int NB = D / 8;
    const int64_t bh = a.bh0 + blockIdx.y;
    uint4 *out = a.frag + ((int64_t)blockIdx.y * a.n_sub + blockIdx.x) * (2 * (D / 16) * kWave);
#pragma unroll
    for (int i = 0; i < 32 * NB / 256; ++i) {
        const int e = threadIdx.x + 256 * i, l32 = e & 31, blk = e >> 5;
        const int64_t t = (int64_t)blockIdx.x * 32 + l32;
        if (t >= a.t_kv) continue;  // masked by the attention kernel
        uint4 hi, lo;
        if (t >= a.t_raw0) {
            const uint4 *kr = reinterpret_cast<const uint4 *>(a.kraw + (bh * a.n_raw + t - a.t_raw0) * 2 * D);
            hi = kr[blk];
            lo = kr[NB + blk];
        } else {
            const int c = a.idx[(bh * a.cap + t) * NB + blk];
            const uint4 *tile = a.codebook + (int64_t)((blk >> 2) * a.nct + (c >> 4)) * 2 * kWave;
            const int l = ((blk & 3) << 4) | (c & 15);
            hi = tile[l];
            lo = __builtin_bit_cast(uint4, __builtin_bit_cast(pg_f16x8, tile[kWave + l]) *
                                               (_Float16)(1.f / 2048.f));
        }
        const int pos = (blk >> 1) * kWave + (blk & 1) * 32 + l32;
        out[pos] = hi;
        out[(D / 16) * kWave + pos] = lo;
    }
}

// LDS plan of prefill_frag_kernel: kStages tiles of KW sub-tiles, each the key
// fragments and then the values (4 blocks of 8 tokens) of 32 tokens.
template <int D, int RW, int KW>
struct FragLds {
    static constexpr int kKeys = 2 * (D / 16) * 1024;
    static constexpr int kSub = kKeys + 32 * D * 2;
    static constexpr int kTile = KW * kSub;
    static constexpr int kStages = KW * D >= 256 ? 3 : 4;
    static constexpr int kPieces = kTile / 1024;                     // 1 KB copies of a tile
    static constexpr int kCopies = (kPieces + RW * KW - 1) / (RW * KW);  // of a wave
    static constexpr int kMerge = KW > 1 ? RW * (D / 32 * 16 + 2) * kWave * 4 : 0;
    static constexpr int kQuery = RW * KW * 32 * (D + 2) * 2;
    static constexpr int kBytes = std::max(kStages * kTile, std::max(kMerge, kQuery));
    static_assert(kBytes <= 160 * 1024, "LDS of a compute unit");
};

enum FragP { kOnePart = 0, kTwoParts = 1, kBf16Parts = 2 };

template <int D, int RW, int KW, int P>
__global__ void __launch_bounds__(RW *KW *kWave, 2) prefill_frag_kernel(FragArgs a) {
    using L = FragLds<D, RW, KW>;
    constexpr bool BF = P == kBf16Parts;
    constexpr int KS = D / 16, NT = D / 32, NW = RW * KW, ROWS = 32 * RW;
    extern __shared__ __align__(16) float4 pg_smem[];
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(pg_smem));
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rw = wv % RW, kg = wv / RW;
    const int hb = lane >> 5, l32 = lane & 31;
    // the longest causal ranges first: row tiles in reverse order
    const int64_t row0 = (int64_t)(a.n_rt - 1 - (int)blockIdx.y) * ROWS;
    const int64_t bh = a.bh0 + blockIdx.x;
    const int64_t bb = bh / a.n_kv_heads;
    const int kvh = (int)(bh - bb * a.n_kv_heads);
    const int64_t n_rows = a.t_q * a.rep;

    // The wave's 32 query rows: round_to(q_dtype, q * scale) (attention.py:208),
    // scaled per row by the power of two that brings its largest element into
    // [2^14, 2^15) (exact in fp16 for fp16 and bf16 elements, down to 2^-29 of
    // the largest; the exponent below takes it back), into LDS as they come
    // (16-byte loads, all in flight), then gathered through the codec's
    // permutation.  (Element loads through the permutation, as prefill32 has
    // them, are 128 dependent round trips: 40 us of every workgroup.)
    constexpr int LPR = D / 8;                 // lanes of a row
    constexpr int RPL = kWave / LPR;           // rows of one pass
    constexpr int kQStride = D + 2;            // halves: a row starts one bank after the one above
    _Float16 *ql = reinterpret_cast<_Float16 *>(pg_smem) + wv * 32 * kQStride;
    const int64_t row = row0 + rw * 32 + l32;
    const bool rok = row < n_rows;
    const int64_t pos = (rok ? row : row0) / a.rep;
    int4 pv[KS][2];  // permutation entries of the lane's dims 16 ks + 8 hb ..
    if (a.perm) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                pv[ks][e] = make_int4(a.perm[16 * ks + 8 * hb + 4 * e], a.perm[16 * ks + 8 * hb + 4 * e + 1],
                                      a.perm[16 * ks + 8 * hb + 4 * e + 2], a.perm[16 * ks + 8 * hb + 4 * e + 3]);
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int j = 16 * ks + 8 * hb + 4 * e;
                pv[ks][e] = make_int4(j, j + 1, j + 2, j + 3);
            }
    }
    int qshift = 0;  // of row l32
    {
        const bool vec = (uintptr_t)a.q % 16 == 0;
        uint4 qr[32 / RPL];
        const int rl = lane / LPR, ch = lane % LPR;
#pragma unroll
        for (int i = 0; i < 32 / RPL; ++i) {
            const int64_t rr = min(row0 + rw * 32 + i * RPL + rl, n_rows - 1);
            const int64_t pp = rr / a.rep;
            const int hh = (int)(rr - pp * a.rep);
            const int64_t off =
                ((bb * a.n_q_heads + (int64_t)kvh * a.rep + hh) * a.t_q + pp) * D + ch * 8;
            const uint16_t *src = static_cast<const uint16_t *>(a.q) + off;
            if (vec) {
                qr[i] = *reinterpret_cast<const uint4 *>(src);
            } else {
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = (uint32_t)src[2 * e] | ((uint32_t)src[2 * e + 1] << 16);
                qr[i] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
#pragma unroll
        for (int i = 0; i < 32 / RPL; ++i) {
            const uint32_t w[4] = {qr[i].x, qr[i].y, qr[i].z, qr[i].w};
            float x[8];
            float mx = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t hw = e & 1 ? w[e / 2] >> 16 : w[e / 2] & 0xffffu;
                const float v = a.q_dtype == SS_F16 ? __half2float(__ushort_as_half((unsigned short)hw))
                                                    : __uint_as_float(hw << 16);
                x[e] = round_to(a.q_dtype, v * a.scale);
                mx = fmaxf(mx, fabsf(x[e]));
            }
#pragma unroll
            for (int o = LPR / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
            const int sh = row_exp_shift(mx);
            const float qinv = exp2i(-sh);
            _Float16 *dst = ql + (i * RPL + rl) * kQStride + ch * 8;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const pg_f16x2 hv = {(_Float16)(x[e] * qinv), (_Float16)(x[e + 1] * qinv)};
                *reinterpret_cast<pg_f16x2 *>(dst + e) = hv;
            }
            const int mine = __shfl(sh, (l32 % RPL) * LPR);
            qshift = l32 / RPL == i ? mine : qshift;
        }
    }
    wave_lds_sync();
    pg_f16x8 qh[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int p8[8] = {pv[ks][0].x, pv[ks][0].y, pv[ks][0].z, pv[ks][0].w,
                           pv[ks][1].x, pv[ks][1].y, pv[ks][1].z, pv[ks][1].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) qh[ks][e] = ql[l32 * kQStride + min(max(p8[e], 0), D - 1)];
    }
    __syncthreads();  // the query rows' LDS becomes the key tiles'
    const float mul = *a.cb_mul * kLog2e * exp2i(qshift);
    const float inv_cb_mul = 1.f / *a.cb_mul;  // a power of two

    // token indices are 32-bit (checked on the host)
    const int64_t row_last = min(row0 + ROWS, n_rows) - 1;
    const int t_end = (int)(a.causal ? min(a.t_kv, a.q_offset + row_last / a.rep + 1) : a.t_kv);
    const int lim = (!rok || !a.causal) ? 0x7fffffff : (int)(a.q_offset + pos);
    // the wave's smallest limit (no mask below it) and the end of what any of
    // its rows sees (nothing to do from there on)
    const int64_t wrow0 = min(row0 + rw * 32, n_rows - 1), wrow1 = min(row0 + rw * 32 + 31, n_rows - 1);
    const int lim_min = a.causal ? (int)(a.q_offset + wrow0 / a.rep) : 0x7fffffff;
    const int w_end = row0 + rw * 32 >= n_rows ? 0
                      : a.causal ? min(t_end, (int)(a.q_offset + wrow1 / a.rep) + 1) : t_end;
    const int n_tiles = (t_end + 32 * KW - 1) / (32 * KW);
    const int blk_last = max(t_end - 1, 0) >> 3;
    const int t_raw0 = a.kraw ? (int)a.t_raw0 : 0x7fffffff;
    const float *kfac = a.kfac + bh * a.n_raw;
    const char *kf = reinterpret_cast<const char *>(a.frag) + (int64_t)blockIdx.x * a.n_sub * L::kKeys;
    const char *v_head = static_cast<const char *>(a.v8) + bh * a.cap_v * D * 2;

    float m = -1e30f, lsum = 0.f;  // row l32 (lsum: this lane half's tokens)
    pg_f32x16 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[nt][i] = 0.f;

    // Tile `tile` into stage `st`, this wave's share of its 1 KB pieces (past
    // the last piece it repeats one, past the last tile the last tile, so
    // every wave always has the same number of copies in flight); value
    // blocks past the last key clamp to its block (zeroed below).
    const uint32_t lane16 = (uint32_t)lane * 16u;
    auto copy_tile = [&](int tile, int st) {
        // (uniform bases and one 32-bit lane offset)
        const int tc = min(tile, n_tiles - 1);
        const char *kb = kf + (uint32_t)tc * (uint32_t)(KW * L::kKeys);
#pragma unroll
        for (int i = 0; i < L::kCopies; ++i) {
            const int piece = min(wv + i * NW, L::kPieces - 1);
            const int sub = piece / (L::kSub / 1024), in = piece % (L::kSub / 1024);
            constexpr int PB = D / 64;  // pieces of an 8-token block
            const int vp = in - L::kKeys / 1024;
            const char *src = in < L::kKeys / 1024
                                  ? kb + (uint32_t)(sub * L::kKeys + in * 1024)
                                  : v_head + (uint32_t)(min((tc * KW + sub) * 4 + vp / PB, blk_last) * PB + vp % PB) *
                                                 1024u;
            __builtin_amdgcn_global_load_lds(
                src + lane16,
                reinterpret_cast<pg_lds<void> *>(lds0 + (uint32_t)(st * L::kTile + piece * 1024)), 16, 0, 0);
        }
    };
    // the tile after the current one has landed (the kStages - 2 after it may
    // still be in flight), for every wave
    auto barrier = [] {
        pg_wait_vm<(L::kStages - 2) * L::kCopies>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (n_tiles > 0) {
#pragma unroll
        for (int i = 0; i < L::kStages - 1; ++i) copy_tile(i, i);
        barrier();
    }
    int stage = 0;
    for (int tile = 0; tile < n_tiles; ++tile) {
        const int t0 = (tile * KW + kg) * 32;
        const uint32_t sub_l = lds0 + (uint32_t)(stage * L::kTile + kg * L::kSub);
        // the stage of the tile before this one takes the tile kStages - 1 on
        const int free_st = stage == 0 ? L::kStages - 1 : stage - 1;
        stage = stage + 1 == L::kStages ? 0 : stage + 1;
        if (t0 >= w_end) {  // past this wave's rows (wave-uniform): copy and meet the others
            copy_tile(tile + L::kStages - 1, free_st);
            barrier();
            continue;
        }
        // key operands in groups of four k-steps, every read of a group in
        // flight before its products (the scheduling barriers keep the
        // compiler from pairing each read with its product, one LDS round
        // trip per product)
        pg_f32x16 sv;
#pragma unroll
        for (int i = 0; i < 16; ++i) sv[i] = 0.f;
        const pg_lds<pg_f16x8> *kt = reinterpret_cast<const pg_lds<pg_f16x8> *>(sub_l) + lane;
        pg_f16x8 kop[KS][2];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < KS; g += 4) {
#pragma unroll
            for (int ks = g; ks < g + 4; ++ks) {
                kop[ks][0] = kt[ks * kWave];
                kop[ks][1] = kt[(KS + ks) * kWave];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            sv = __builtin_amdgcn_mfma_f32_32x32x16_f16(kop[ks][0], qh[ks], sv, 0, 0, 0);
            sv = __builtin_amdgcn_mfma_f32_32x32x16_f16(kop[ks][1], qh[ks], sv, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // value operands: 4 tokens of one dim (8 bytes) for 4 steps of 8
        // tokens and NT tiles of 32 dims
        pg_u32x2 vop[4][NT];
        const pg_lds<pg_u32x2> *vt =
            reinterpret_cast<const pg_lds<pg_u32x2> *>(sub_l + L::kKeys) + 2 * l32 + hb;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) vop[kk][nt] = vt[(kk * D + nt * 32) * 2];
        __builtin_amdgcn_sched_barrier(0);
        // (after the tile's LDS reads)
        copy_tile(tile + L::kStages - 1, free_st);
        if (t0 + 31 >= t_raw0) {  // whole keys carry their own power of two
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int tk = t0 + 8 * (i >> 2) + 4 * hb + (i & 3);
                if (tk >= t_raw0 && tk < t_end) sv[i] *= kfac[tk - t_raw0] * inv_cb_mul;
            }
        }
        if (!(t0 + 31 < t_end && t0 + 31 <= lim_min)) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int tk = t0 + 8 * (i >> 2) + 4 * hb + (i & 3);
                sv[i] = (tk < t_end && tk <= lim) ? sv[i] : -INFINITY;
            }
        }
        // online softmax of row l32 (16 of its 32 tokens here, 16 in lane ^ 32)
        float mx = sv[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = fmaxf(mx, sv[i]);
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = (mx - m) * mul > kPgLag ? fmaxf(m, mx) : m;
        const float corr = fast_exp2((m - mn) * mul);
        m = mn;
        float ps = 0.f;
        const float off = fmaf(mn, mul, -kPgExp);
        uint32_t ph[8], pl[P != kOnePart ? 8 : 1], pm[BF ? 8 : 1];  // pairs of tokens: the operand's parts
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const float x0 = fast_exp2(fmaf(sv[i], mul, -off));
            const float x1 = fast_exp2(fmaf(sv[i + 1], mul, -off));
            ps += x0;
            ps += x1;
            if constexpr (BF) {
                // truncated parts, all above zero where the probability is
                // (the factor leaves each at least x * 2^-23 to take, an ulp of
                // the probability at most): a part that is zero or negative,
                // as rounded ones are, would make NaN of an infinite value
                const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
                ph[i / 2] = pg_high_halves(u0, u1);
                const float r0 = fmaf(x0, kPgMore, -__uint_as_float(u0 & 0xffff0000u));
                const float r1 = fmaf(x1, kPgMore, -__uint_as_float(u1 & 0xffff0000u));
                const uint32_t w0 = __float_as_uint(r0), w1 = __float_as_uint(r1);
                pl[i / 2] = pg_high_halves(w0, w1);
                pm[i / 2] = pg_high_halves(
                    __float_as_uint(fmaf(r0, kPgMore, -__uint_as_float(w0 & 0xffff0000u))),
                    __float_as_uint(fmaf(r1, kPgMore, -__uint_as_float(w1 & 0xffff0000u))));
            } else {
                const pg_f16x2 hi = __builtin_convertvector((pg_f32x2){x0, x1}, pg_f16x2);
                ph[i / 2] = __builtin_bit_cast(uint32_t, hi);
                if constexpr (P == kTwoParts)
                    pl[i / 2] = __builtin_bit_cast(
                        uint32_t, __builtin_convertvector((pg_f32x2){x0 - (float)hi[0], x1 - (float)hi[1]}, pg_f16x2));
            }
        }
        lsum = fmaf(lsum, corr, ps);
        if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0) {
            // accumulator rows 8 (i/4) + 4 hb + i%4: their own rows' correction
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float ci = pg_lane(corr, 8 * (i >> 2) + 4 * hb + (i & 3));
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[nt][i] *= ci;
            }
        }
        if (t0 + 32 > t_end) {
            // zero the values of tokens past the last key (their weights are
            // zero, what lies there need not be finite)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int n_ok = max(min(t_end - (t0 + 8 * kk + 4 * hb), 4), 0);
                const uint32_t zx = n_ok >= 2 ? 0xffffffffu : n_ok == 1 ? 0x0000ffffu : 0u;
                const uint32_t zy = n_ok >= 4 ? 0xffffffffu : n_ok == 3 ? 0x0000ffffu : 0u;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    vop[kk][nt].x &= zx;
                    vop[kk][nt].y &= zy;
                }
            }
        }
        // step k2: the lane's eight tokens are entries 8 k2 .. +7 (tokens
        // 16 k2 + 4 hb + 0..3 and 16 k2 + 8 + 4 hb + 0..3), in A and in B
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2) {
            const uint4 ah = make_uint4(ph[4 * k2], ph[4 * k2 + 1], ph[4 * k2 + 2], ph[4 * k2 + 3]);
            uint4 al = ah, am = ah;
            if constexpr (P != kOnePart)
                al = make_uint4(pl[4 * k2], pl[4 * k2 + 1], pl[4 * k2 + 2], pl[4 * k2 + 3]);
            if constexpr (BF)
                am = make_uint4(pm[4 * k2], pm[4 * k2 + 1], pm[4 * k2 + 2], pm[4 * k2 + 3]);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const uint4 b = make_uint4(vop[2 * k2][nt].x, vop[2 * k2][nt].y, vop[2 * k2 + 1][nt].x,
                                           vop[2 * k2 + 1][nt].y);
                if constexpr (BF) {
                    acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(pg_bf16x8, am), __builtin_bit_cast(pg_bf16x8, b), acc[nt], 0, 0, 0);
                    acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(pg_bf16x8, al), __builtin_bit_cast(pg_bf16x8, b), acc[nt], 0, 0, 0);
                    acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(pg_bf16x8, ah), __builtin_bit_cast(pg_bf16x8, b), acc[nt], 0, 0, 0);
                } else {
                    acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        __builtin_bit_cast(pg_f16x8, ah), __builtin_bit_cast(pg_f16x8, b), acc[nt], 0, 0, 0);
                    if constexpr (P == kTwoParts)
                        acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            __builtin_bit_cast(pg_f16x8, al), __builtin_bit_cast(pg_f16x8, b), acc[nt], 0, 0, 0);
                }
            }
        }
        barrier();
    }

    // the KW partial softmaxes of a row meet in LDS, key group 0 takes the
    // others' in turn: [RW][NT*16 + 2][64 lanes] floats
    pg_wait_vm<0>();  // (the last copies repeat the last tile)
    float Ls = lsum + __shfl_xor(lsum, 32);
    float *part = reinterpret_cast<float *>(pg_smem) + rw * (NT * 16 + 2) * kWave + lane;
#pragma unroll 1
    for (int g = 1; g < KW; ++g) {
        __syncthreads();  // (the first: every wave is done with the key tiles)
        if (kg == g) {
            part[0] = m;
            part[kWave] = Ls;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 16; ++i) part[(2 + nt * 16 + i) * kWave] = acc[nt][i];
        }
        __syncthreads();
        if (kg == 0) {
            const float m2 = part[0], L2 = part[kWave];
            const float mn = fmaxf(m, m2);
            const float f1 = fast_exp2((m - mn) * mul), f2 = fast_exp2((m2 - mn) * mul);
            m = mn;
            Ls = Ls * f1 + L2 * f2;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int ri = 8 * (i >> 2) + 4 * hb + (i & 3);
                const float c1 = pg_lane(f1, ri), c2 = pg_lane(f2, ri);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acc[nt][i] = acc[nt][i] * c1 + part[(2 + nt * 16 + i) * kWave] * c2;
            }
        }
    }
    if (kg != 0) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int ri = 8 * (i >> 2) + 4 * hb + (i & 3);
        const float Li = pg_lane(Ls, ri);
        const int64_t orow = row0 + rw * 32 + ri;
        if (orow < n_rows) {
            const int64_t op = orow / a.rep;
            const int oh = (int)(orow - op * a.rep);
            const int64_t off = ((bb * a.n_q_heads + (int64_t)kvh * a.rep + oh) * a.t_q + op) * D;
            // acc and l both carry 2^11 (bfloat16 parts: acc an ulp more)
            const float inv = Li > 0.f ? (BF ? 2.f - kPgMore : 1.f) / Li : 0.f;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                store_from_f32(a.out, a.out_dtype, off + 32 * nt + l32, acc[nt][i] * inv);
        }
    }
}

// Sub-tiles of a head's fragments (whole tiles of the largest KW).
static int64_t frag_subs(int64_t t_kv) { return (t_kv + 63) / 64 * 2; }
static int64_t frag_head_bytes(int64_t t_kv, int d) { return frag_subs(t_kv) * 32 * d * 4; }
// Fragments beyond this many bytes are built and used a few heads at a time.
constexpr int64_t kFragBytes = int64_t(256) << 20;

template <int D, int RW, int KW, int P>
static int launch_frag(const FragArgs &a, int64_t n_bh, hipStream_t st) {
    constexpr int lds = FragLds<D, RW, KW>::kBytes;
    auto kern = prefill_frag_kernel<D, RW, KW, P>;
    static bool attr_set = false;
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(prefill frag)");
        attr_set = true;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)n_bh, a.n_rt), dim3(RW * KW * kWave), lds, st, a);
    SS_LAUNCH_CHECK("prefill_frag_kernel launch");
    return SS_OK;
}

}  // namespace ss

using namespace ss;

extern "C" size_t ss_prefill_workspace_bytes(int64_t batch, int n_kv_heads, int head_dim,
                                             int64_t t_kv) {
    if (batch < 1 || n_kv_heads < 1 || t_kv < 1) return 0;
    const int64_t head = frag_head_bytes(t_kv, head_dim);
    return (size_t)std::max(head, std::min(batch * n_kv_heads * head, kFragBytes / head * head));
}

extern "C" int ss_prefill_attn(const void *q, int q_dtype, int64_t batch, int n_q_heads,
                               int n_kv_heads, int64_t t_q, int head_dim, float scale,
                               const int32_t *perm, const void *codebook, int n_blocks,
                               int n_centroids, const uint8_t *idx, int64_t cap,
                               const void *values_il8, int v_dtype, int64_t cap_v, int64_t t_kv,
                               const void *kraw, const float *kfac, int64_t t_raw0, int causal,
                               int64_t q_offset, void *out, int out_dtype, void *workspace,
                               size_t workspace_bytes, void *stream) {
    SS_REQUIRE(q && codebook && idx && values_il8 && out, "null pointer argument");
    SS_REQUIRE(valid_dtype(q_dtype) && valid_dtype(out_dtype), "bad dtype code");
    SS_REQUIRE(batch >= 1 && n_q_heads >= 1 && n_kv_heads >= 1 && t_q >= 1 &&
                   n_q_heads % n_kv_heads == 0, "bad head/batch counts");
    SS_UNSUPPORTED((head_dim == 64 || head_dim == 128) && n_blocks * 8 == head_dim,
                   "prompt kernel takes head_dim 64 or 128 in blocks of 8 (got %d, %d blocks)",
                   head_dim, n_blocks);
    SS_UNSUPPORTED(n_centroids >= 1 && n_centroids <= 256, "n_centroids %d unsupported (1..256)",
                   n_centroids);
    SS_UNSUPPORTED(q_dtype == SS_F16 || q_dtype == SS_BF16, "prompt kernel takes fp16 or bf16 queries");
    SS_UNSUPPORTED(v_dtype == SS_F16 || v_dtype == SS_BF16,
                   "interleaved values must be float16 or bfloat16");
    SS_REQUIRE(cap_v % 8 == 0 && t_kv >= 1 && t_kv <= cap_v,
               "bad cap/t_kv (the value capacity a multiple of 8, 1 <= t_kv <= it)");
    const bool raw = kraw != nullptr;
    SS_REQUIRE(!raw || (kfac && t_raw0 >= 0 && t_raw0 <= t_kv && t_raw0 <= cap),
               "whole keys need their factors and 0 <= t_raw0 <= min(t_kv, cap)");
    SS_REQUIRE(raw || t_kv <= cap, "t_kv exceeds the index capacity");
    SS_REQUIRE(q_offset >= 0, "negative q_offset");
    SS_UNSUPPORTED(cap_v < (int64_t(1) << 23) && t_q + q_offset < (int64_t(1) << 30),
                   "prompt kernel takes caches below 2^23 tokens");
    SS_REQUIRE(((uintptr_t)codebook % 16) == 0 && ((uintptr_t)values_il8 % 16) == 0 &&
                   ((uintptr_t)kraw % 16) == 0 && ((uintptr_t)workspace % 16) == 0,
               "codebook, values, whole keys and workspace must be 16-byte aligned");
    const int64_t head = frag_head_bytes(t_kv, head_dim), n_bh = batch * n_kv_heads;
    const int64_t per = std::min<int64_t>((int64_t)(workspace_bytes / head), std::min<int64_t>(n_bh, 65535));
    if (!workspace || per < 1) {
        set_error("prompt workspace too small: one head needs %lld bytes, got %zu", (long long)head,
                  workspace ? workspace_bytes : (size_t)0);
        return SS_ERR_WORKSPACE;
    }
    FragArgs a;
    a.q = q;
    a.q_dtype = q_dtype;
    a.n_q_heads = n_q_heads;
    a.n_kv_heads = n_kv_heads;
    a.rep = n_q_heads / n_kv_heads;
    a.t_q = t_q;
    a.scale = scale;
    a.perm = perm;
    a.codebook = static_cast<const uint4 *>(codebook);
    a.nct = (n_centroids + 15) / 16;
    a.cb_mul = reinterpret_cast<const float *>(static_cast<const char *>(codebook) +
                                               (size_t)(n_blocks / 4) * a.nct * 2 * kWave * 16);
    a.idx = idx;
    a.v8 = values_il8;
    a.cap = cap;
    a.cap_v = cap_v;
    a.t_kv = t_kv;
    a.kraw = static_cast<const __half *>(kraw);
    a.kfac = kfac;
    a.t_raw0 = raw ? t_raw0 : t_kv;
    a.n_raw = raw ? std::max<int64_t>(t_kv - t_raw0, 1) : 0;
    a.causal = causal ? 1 : 0;
    a.q_offset = q_offset;
    a.out = out;
    a.out_dtype = out_dtype;
    a.frag = static_cast<uint4 *>(workspace);
    a.n_sub = frag_subs(t_kv);
    // Waves of a workgroup.  8 x 1 (256 rows, every wave on the same tile)
    // streams a tile for the most rows and is the fastest per row where it
    // fills the chip evenly; 4 x 2 (128 rows, two key groups) gives twice
    // the workgroups.  head_dim 128, 32/8 heads, us (8 x 1 / 4 x 2): 4096 new
    // tokens 258 / 318, 2048 new 118 / 106 (one workgroup a compute unit, of
    // uneven causal ranges), 2048 after 32768 1799 / 1934, 4 x 512 after 4096
    // 274 / 308, 2 x 512 after 8192 421 / 280.  head_dim 64 has room for two
    // workgroups on a compute unit, so 4 x 1 takes that place (4 x 1 / 4 x 2):
    // 149 / 198, 67 / 67, 1111 / 1146, 178 / 206, 239 / 179.
    const int64_t cus = device_cu_count();
    const int64_t n256 = (t_q * a.rep + 255) / 256 * n_bh, n128 = (t_q * a.rep + 127) / 128 * n_bh;
    const bool wide = head_dim == 128
                          ? n256 >= 2 * cus || (n256 >= cus && (!causal || q_offset >= t_q))
                          : n128 >= 2 * cus;
    const int RW = wide && head_dim == 128 ? 8 : 4;
    const int64_t n_rt = (t_q * a.rep + 32 * RW - 1) / (32 * RW);
    SS_UNSUPPORTED(n_rt <= 65535, "grid too large");
    a.n_rt = (int)n_rt;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // fp16 probabilities: one part (11 bits) for prompts of at least 128 rows at
    // head_dim 128 in whole GQA groups, where the second product would cost a
    // fifth of the time and one part keeps the output within 4.1e-4 of its
    // largest value at 4096 tokens; two parts for the calls whose other
    // kernel, a decode, has 22-bit probabilities too.
    const int parts = v_dtype == SS_BF16 ? kBf16Parts
                      : head_dim == 128 && 128 % a.rep == 0 && t_q * a.rep >= 128 ? kOnePart : kTwoParts;
    for (int64_t bh0 = 0; bh0 < n_bh; bh0 += per) {
        const int64_t n = std::min(per, n_bh - bh0);
        a.bh0 = bh0;
        const dim3 kg((unsigned)((t_kv + 31) / 32), (unsigned)n);
        if (head_dim == 128)
            hipLaunchKernelGGL(prefill_keys_kernel<128>, kg, dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL(prefill_keys_kernel<64>, kg, dim3(256), 0, st, a);
        SS_LAUNCH_CHECK("prefill_keys_kernel launch");
#define SS_FRAG(DD, RR, KK)                                                        \
    (parts == kBf16Parts  ? launch_frag<DD, RR, KK, kBf16Parts>(a, n, st)           \
     : parts == kTwoParts ? launch_frag<DD, RR, KK, kTwoParts>(a, n, st)            \
                          : launch_frag<DD, RR, KK, DD == 128 ? kOnePart : kTwoParts>(a, n, st))
        const int rc = head_dim == 128 ? (wide ? SS_FRAG(128, 8, 1) : SS_FRAG(128, 4, 2))
                                       : (wide ? SS_FRAG(64, 4, 1) : SS_FRAG(64, 4, 2));
#undef SS_FRAG
        if (rc) return rc;
    }
    return SS_OK;
}
