// FLASH_ATTN_EXT for many query rows (prefill) on the f16 matrix cores.
// Semantics: ggml_compute_forward_flash_attn_ext_f16, ggml/src/ggml-cpu/ggml-cpu.c:10916-11129
// (q rounded to f16, scores scale * q.k [+ softcap] + slope * mask, online softmax in f32,
// -inf mask entries contribute nothing, GQA by head index division).
//
// A 256-thread group serves one kv head: its 4 waves are HPW query heads of that kv head times
// 4 / HPW tiles of 32 queries, so every K/V tile staged in LDS is used by all four waves.
// Per wave and 64-cell kv tile, with v_mfma_f32_32x32x16_f16 (D[i][j], lane l supplies row /
// column l % 32 and k slots [8*(l/32), +8); D register r is i = 8*(r/4) + 4*(l/32) + r%4, j = l%32):
//   S^T = K Q^T   A = K rows (i = kv cell), B = Q rows (j = query)  -> a lane holds ONE query's
//                 scores for 16 cells, so softmax row reductions are in-lane plus one xor-32 step
//   O^T += V^T P^T  A = V^T rows (i = head dim), B = P^T (j = query) -> the B operand is the lane's
//                 own score registers 8t..8t+7 rounded to f16: no cross-lane data movement.  The
//                 kv cells those registers stand for, 16t + 8*(s/4) + 4*(l/32) + s%4, fix which
//                 cells the A operand must supply in k slot s: four cells at one element of the head, twice -
//                 two transposing reads (ds_read_b64_tr_b16) of the row-major V tile.
// Rescaling by exp(m_old - m_new) is one multiply per accumulator register because both
// accumulators are indexed by query along the lanes.
#include "fattn.hpp"


#include <float.h>

namespace mi355 {

namespace {

constexpr int FM_BC = 64;            // kv cells per tile
constexpr float FM_NEG = -FLT_MAX / 2;

// O^T is accumulated in tiles of 32 elements of the head: head sizes that are no multiple of 32 (80, 112) leave the last tile partly
// unused - its upper rows meet whatever the padding columns of the V tile hold and are never stored.
template <int D> constexpr int fm_dtiles() { return (D + 31) / 32; }
template <int D> constexpr int fm_vpitch() { return 32 * fm_dtiles<D>() + 16; }   // f16 pitch of a V row in LDS: rows 8 banks apart, so the four rows of a transposing read miss each other

// ---- staging of one 64-cell K tile and the matching V tile through registers, both row-major ----
template <int D, int NTH, int BC = FM_BC> struct kv_stage {
    static constexpr int KP = D + 8;        // f16 pitch of a K row in LDS (16 bytes of padding spread the banks)
    static constexpr int VP = fm_vpitch<D>();
    static constexpr int KCH = D / 8;       // 16-byte chunks per K/V row
    static constexpr int UNITS = BC * KCH;
    static constexpr int KIT = (UNITS + NTH - 1) / NTH;   // chunks per thread per tile, K and V each
    static constexpr bool EVEN = NTH % KCH == 0 && UNITS % NTH == 0;   // a thread keeps its chunk position over the rows it loads
    static_assert(D % 16 == 0, "head size not served by this kernel");
    u32x4 k[KIT], v[KIT];

    // A tile that lies inside the cache is addressed as (uniform base of the tile and of the thread's it-th row block) + (one
    // 32-bit offset per thread, the same for every tile): thread tid loads rows tid / KCH + it * (NTH / KCH), chunk tid % KCH.
    // The uniform part is scalar arithmetic; per-row 64-bit products in vector registers cost as many instructions per tile
    // step as the soft-max.  The launcher checks that a tile's span fits 32 bits.  Head sizes whose chunks do not divide the group
    // evenly (80, 96, 112) keep one offset per chunk instead.  The last, partial tile clamps row by row.
    __device__ __forceinline__ void fetch(const fattn_args &a, int64_t hk, int64_t kv0, int tid) {
        if (kv0 + BC <= a.Nkv) {   // uniform
            const uint8_t *kb = a.k + kv0 * a.k_nb1 + hk * a.k_nb2, *vb = a.v + kv0 * a.v_nb1 + hk * a.v_nb2;
            if constexpr (EVEN) {
                const unsigned r0 = (unsigned)(tid / KCH), ch16 = (unsigned)(tid % KCH) * 16;
                const unsigned ko = r0 * (unsigned)a.k_nb1 + ch16, vo = r0 * (unsigned)a.v_nb1 + ch16;
#pragma unroll
                for (int it = 0; it < KIT; it++) {
                    k[it] = load16(kb + (size_t)it * (NTH / KCH) * a.k_nb1 + ko);
                    v[it] = load16(vb + (size_t)it * (NTH / KCH) * a.v_nb1 + vo);
                }
            } else {
#pragma unroll
                for (int it = 0; it < KIT; it++) {
                    const unsigned unit = tid + it * NTH < UNITS ? tid + it * NTH : UNITS - 1;
                    const unsigned row = unit / KCH, ch16 = unit % KCH * 16;
                    k[it] = load16(kb + (row * (unsigned)a.k_nb1 + ch16));
                    v[it] = load16(vb + (row * (unsigned)a.v_nb1 + ch16));
                }
            }
            return;
        }
        const int64_t last = a.Nkv - 1;
#pragma unroll
        for (int it = 0; it < KIT; it++) {
            const int unit = EVEN || tid + it * NTH < UNITS ? tid + it * NTH : UNITS - 1;
            const int row = unit / KCH, ch = unit % KCH;
            const int64_t c = kv0 + row < last ? kv0 + row : last;   // rows past the end repeat the last cell; their scores are dropped
            k[it] = load16(a.k + c * a.k_nb1 + hk * a.k_nb2 + ch * 16);
            v[it] = load16(a.v + c * a.v_nb1 + hk * a.v_nb2 + ch * 16);
        }
    }
    __device__ __forceinline__ void commit(_Float16 *sK, _Float16 *sV, int tid) const {
#pragma unroll
        for (int it = 0; it < KIT; it++) {
            const int unit = tid + it * NTH;
            if (UNITS % NTH != 0 && unit >= UNITS) continue;
            const int row = unit / KCH, ch = unit % KCH;
            *(u32x4 *)(sK + row * KP + ch * 8) = k[it];
            *(u32x4 *)(sV + row * VP + ch * 8) = v[it];
        }
    }
};

// f16 bits of the mask entries of NG groups of 4 consecutive cells, first cell c0 + 8*g.  Loads are
// unconditional (clamped), so they can be issued with the K/V prefetch and never force a wait.
template <int NG>
__device__ __forceinline__ void fetch_mask(u32x2 (&out)[NG], const unsigned short *mrow, bool vec_ok, int64_t c0, int64_t Nkv) {
    if (mrow == nullptr) {
#pragma unroll
        for (int g = 0; g < NG; g++) out[g] = u32x2{0, 0};
    } else if (vec_ok) {   // uniform: aligned rows and a full tile
#pragma unroll
        for (int g = 0; g < NG; g++) out[g] = *(const u32x2 *)(mrow + c0 + 8 * g);
    } else {
        const int64_t last = Nkv - 1;
#pragma unroll
        for (int g = 0; g < NG; g++) {
            u32 h[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int64_t c = c0 + 8 * g + i;
                h[i] = mrow[c < last ? c : last];
            }
            out[g] = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
        }
    }
}
__device__ __forceinline__ float mask_value(const u32x2 &w, int i) {
    return half_bits_to_float((unsigned short)((i < 2 ? w[0] : w[1]) >> (16 * (i & 1))));
}

// max / sum of a value over a lane and its partner in the other half of the wave (lane ^ 32), in every lane: one
// v_permlane32_swap (both halves of one register handed to the other half of a second) instead of a trip through the LDS
// crossbar, whose latency a wave that is alone on its SIMD waits out.
__device__ __forceinline__ float half_pair_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_pair_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Running maximum of the prefill kernels.  The reference point of a column's exponentials moves only when the tile's largest
// score exceeds it by more than FM_LAZY: any reference point gives the same quotient sum(p v) / sum(p), and while it stays put
// the 64 output registers are not rescaled (with an exact running maximum some query of a 32-query tile raises its maximum
// in most tiles of a few thousand cells; this way it happens in the first tiles only).  Probabilities then reach e^FM_LAZY at
// most, far inside the f16 range of the matrix operand.
constexpr float FM_LAZY = 8.0f;
constexpr float FM_LOG2E = 1.4426950408889634f;
//
// PX: probabilities of f32 precision, for the calls whose other form (the vector kernel) multiplies f32 probabilities: the matrix operand
// is f16, so a probability goes in as 2^10 p = hi + lo, two f16 values, and every V fragment meets two matrix instructions.  The factor
// (exact, taken back at the end) keeps lo of a small probability from being subnormal: with probabilities of at most e^4 (2^10 e^4 < 65504)
// the pair is within 2^-22 p or 2^-35 of one at the reference point.  Error against 64-bit arithmetic and time: see launch_fattn_mma.
constexpr float FM_PX_SCALE = 1024.0f;
template <int D> constexpr int fm_px_chains() { return D == 64 || D == 128 ? 4 : 2; }   // partial sums of a score (one chain: D 128, 512 x 512 cells 1.48e-7, four 1.26e-7; vector kernel 1.28e-7)
template <bool PX> __device__ __forceinline__ float lazy_max(float m, float mx) { return mx > m + (PX ? 4.0f : FM_LAZY) ? mx : m; }
// the reference point as a power of two.  PX: rounded once and used as it is wherever exponents are compared, so that old and new terms of a sum agree
template <bool PX> __device__ __forceinline__ float exponent_of(float m) { return PX ? mul_rn(m, FM_LOG2E) : m * FM_LOG2E; }
// what a state with reference point m is multiplied with when the point moves to m_new
template <bool PX> __device__ __forceinline__ float rescale(float m, float m_new) {
    return PX ? __builtin_amdgcn_exp2f(sub_rn(exponent_of<true>(m), exponent_of<true>(m_new))) : __builtin_amdgcn_exp2f((m - m_new) * FM_LOG2E);
}
// ... and when two finished states are joined
template <bool PX> __device__ __forceinline__ float merge_factor(float m, float M) { return PX ? rescale<true>(m, M) : __expf(m - M); }
// O / sum with inv = reciprocal of the sum.  PX: rounded once (one correction step); a row without a visible cell is 0 / 0, as in the vector kernel
template <bool PX> __device__ __forceinline__ float sum_of(float l) { return PX ? l * FM_PX_SCALE : l; }
template <bool PX> __device__ __forceinline__ float reciprocal_of(float l) { return PX || l > 0.0f ? 1.0f / l : 0.0f; }
template <bool PX> __device__ __forceinline__ float quotient(float o, float l, float inv) {
    const float q = o * inv;
    return PX ? fmaf(fmaf(-q, l, o), inv, q) : q;
}
// exp(s - m) as one multiply-add and one exponential: 2^(s log2(e) - m log2(e)); m2 = m log2(e)
__device__ __forceinline__ float exp_rel(float s, float m2) { return __builtin_amdgcn_exp2f(fmaf(s, FM_LOG2E, -m2)); }

// the larger of two, NaN if one of them is (v_maximum3_f32)
__device__ __forceinline__ float max_or_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float half_pair_max_or_nan(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return max_or_nan(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// scale [+ softcap], add the mask; returns the largest score, NaN if there is one (such a tile is not skipped).  A masked cell (-inf) and one past the end of the range end as -inf, a
// probability of exactly 0.  A NaN stays one and shows in the column's sum (store_rows).  The test against the end of the range is
// made only in a tile that reaches past it (uniform over the group), on 32-bit offsets.
__device__ __forceinline__ float finish_scores(f32x16 &S, const u32x2 (&mw)[4], const fattn_args &a, float scale, float slope,
                                                int64_t c_first, int lhi, int64_t c_end) {
    float mx = FM_NEG;
    const int64_t room = c_end - c_first;
    if (a.softcap == 0.0f && slope == 1.0f && room >= 32) {   // the common case in one multiply-add per score: scale * s + mask
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                S[4 * g + i] = fmaf(S[4 * g + i], scale, mask_value(mw[g], i));
                mx = max_or_nan(mx, S[4 * g + i]);
            }
        return mx;
    }
    if (a.softcap != 0.0f) {
#pragma unroll
        for (int r = 0; r < 16; r++) S[r] = a.softcap * tanhf(S[r] * scale);
    } else {
#pragma unroll
        for (int r = 0; r < 16; r++) S[r] *= scale;
    }
    const int left = room < 32 ? (int)room - 4 * lhi : 32;   // cells of the range from this lane's first one on (may be <= 0)
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float mv = mask_value(mw[g], i);
            S[4 * g + i] = 8 * g + i < left && mv != -INFINITY ? S[4 * g + i] + slope * mv : -INFINITY;
            mx = max_or_nan(mx, S[4 * g + i]);
        }
    return mx;
}
// The decode kernel keeps the plain form (every score tested against the end of its kv range): with its two tile bodies the
// split into a full-tile and an end-of-range variant cost it 10 % at 131072 cells (115 -> 127 us) for 2 % gained at 32768.
__device__ __forceinline__ float finish_scores_dec(f32x16 &S, const u32x2 (&mw)[4], const fattn_args &a, float scale, float slope,
                                                    int64_t c_first, int lhi, int64_t c_end) {
    if (a.softcap != 0.0f) {
#pragma unroll
        for (int r = 0; r < 16; r++) S[r] = a.softcap * tanhf(S[r] * scale);
    } else {
#pragma unroll
        for (int r = 0; r < 16; r++) S[r] *= scale;
    }
    float mx = FM_NEG;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const int64_t c = c_first + 8 * g + 4 * lhi;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float mv = mask_value(mw[g], i);
            float s = S[4 * g + i] + slope * mv;
            const bool valid = c + i < c_end && mv != -INFINITY && s > FM_NEG;   // NaN scores of stale cells drop out too
            s = valid ? s : FM_NEG;
            S[4 * g + i] = s;
            mx = fmaxf(mx, s);
        }
    }
    return mx;
}

// A query row's share of a lane (elements 16 kk + 8 lhi .. + 7), requested ahead of the first K/V tile - loads return in the order of their issue - and rounded to f16
// (ggml-cpu.c:11037-11040) while that tile is on its way
template <int D>
struct q_row {
    f32x4 x[D / 8];
    __device__ __forceinline__ void request(const float *qp, int lhi) {
#pragma unroll
        for (int kk = 0; kk < D / 16; kk++) {
            x[2 * kk] = *(const f32x4 *)(qp + 16 * kk + 8 * lhi);
            x[2 * kk + 1] = *(const f32x4 *)(qp + 16 * kk + 8 * lhi + 4);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void convert(f16x8 (&qf)[D / 16]) const {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < D / 16; kk++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                qf[kk][i] = (_Float16)x[2 * kk][i];
                qf[kk][4 + i] = (_Float16)x[2 * kk + 1][i];
            }
    }
};
__device__ __forceinline__ float alibi_slope(const fattn_args &a, int64_t head) {   // ggml-cpu.c:10998-11003
    if (a.max_bias <= 0.0f) return 1.0f;
    const unsigned h = (unsigned)head;
    return h < a.n_head_log2 ? powf(a.m0, (float)(h + 1)) : powf(a.m1, (float)(2 * (h - a.n_head_log2) + 1));
}

// O^T tiles [DT0, DT0 + NDT) += V^T P^T for the 32 cells of half u whose probabilities sit in S.  The A operand of a lane -
// element 32 dt + l32 of cells c .. c + 3 and c + 8 .. c + 11, c = 32 u + 16 t + 4 lhi - comes from the row-major V tile by two
// transposing reads: in each group of 16 lanes, lane i receives element i % 4 of the four rows that lanes i / 4, i / 4 + 4, + 8 and
// + 12 point at, so lane 4 r + q of a group points at row c + r, elements 16 (group % 2) + 4 q .. + 3 of the tile's 32.
template <int D>
__device__ __forceinline__ const _Float16 *v_lane_base(const _Float16 *sV, int u, int l32, int lhi) {
    const int li = l32 & 15;
    return sV + (32 * u + 4 * lhi + (li >> 2)) * fm_vpitch<D>() + 16 * (l32 >> 4) + 4 * (li & 3);
}
template <int VP>
__device__ __forceinline__ f16x8 v_fragment(const _Float16 *vp) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)vp);
    const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(vp + 8 * VP));
    const f16x4 h0 = __builtin_bit_cast(f16x4, v0), h1 = __builtin_bit_cast(f16x4, v1);
    f16x8 vf;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        vf[i] = h0[i];
        vf[4 + i] = h1[i];
    }
    return vf;
}
template <int D, int NDT>
__device__ __forceinline__ void accumulate_pv(f32x16 (&o)[NDT], const f32x16 &S, const _Float16 *sV, int dt0, int u, int l32, int lhi) {
    constexpr int VP = fm_vpitch<D>();
    const _Float16 *lane_base = v_lane_base<D>(sV, u, l32, lhi);
#pragma unroll
    for (int t = 0; t < 2; t++) {
        f16x8 pf;
#pragma unroll
        for (int i = 0; i < 8; i++) pf[i] = (_Float16)S[8 * t + i];
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_fragment<VP>(lane_base + 16 * t * VP + 32 * (dt0 + dt)), pf, o[dt], 0, 0, 0);
    }
}
// PX: the same for the NS halves u0 .. of a tile, with probabilities as pairs.  A tile's terms are added up from zero and meet the long sum
// once: of the roundings of O those are the ones that count (one per tile of 64 cells where the vector kernel has one per 16 or 32 cells).
template <int D, int NDT, int NS>
__device__ __forceinline__ void accumulate_pv_px(f32x16 (&o)[NDT], const f32x16 (&S)[NS], const _Float16 *sV, int u0, int l32, int lhi) {
    constexpr int VP = fm_vpitch<D>();
    f16x8 hi[2 * NS], lo[2 * NS];
#pragma unroll
    for (int t = 0; t < 2 * NS; t++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float p = S[t / 2][8 * (t & 1) + i];
            hi[t][i] = (_Float16)(p * FM_PX_SCALE);
            lo[t][i] = (_Float16)fmaf(p, FM_PX_SCALE, -(float)hi[t][i]);   // exact before the conversion
        }
    const _Float16 *lane_base = v_lane_base<D>(sV, u0, l32, lhi);
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) {
        f32x16 sum;
#pragma unroll
        for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll
        for (int t = 0; t < 2 * NS; t++) {
            const f16x8 vf = v_fragment<VP>(lane_base + 16 * t * VP + 32 * dt);
            sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, lo[t], sum, 0, 0, 0);
            sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, hi[t], sum, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] += sum[r];
    }
}

// EAGER: all of the row's fragments are requested before the first matrix instruction (D / 2 more registers), so the chain of
// dependent instructions does not stop for an LDS round trip after every second one.
// CHAINS: independent partial sums of D / CHAINS elements each, added at the end (smaller sums, smaller roundings)
template <int D, bool EAGER = false, int CHAINS = 1>
__device__ __forceinline__ f32x16 scores(const f16x8 (&qf)[D / 16], const _Float16 *sK, int u, int l32, int lhi) {
    constexpr int KP = D + 8;
    if constexpr (CHAINS > 1) {
        f32x16 part[CHAINS];
#pragma unroll
        for (int c = 0; c < CHAINS; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) part[c][r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < D / 16; kk++) {
            const f16x8 kf = *(const f16x8 *)(sK + (32 * u + l32) * KP + 16 * kk + 8 * lhi);
            part[kk % CHAINS] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[kk], part[kk % CHAINS], 0, 0, 0);
        }
#pragma unroll
        for (int step = 1; step < CHAINS; step *= 2)
#pragma unroll
            for (int c = 0; c + step < CHAINS; c += 2 * step)
#pragma unroll
                for (int r = 0; r < 16; r++) part[c][r] += part[c + step][r];
        return part[0];
    }
    f32x16 S;
#pragma unroll
    for (int r = 0; r < 16; r++) S[r] = 0.0f;
    if constexpr (EAGER) {
        f16x8 kf[D / 16];
#pragma unroll
        for (int kk = 0; kk < D / 16; kk++) kf[kk] = *(const f16x8 *)(sK + (32 * u + l32) * KP + 16 * kk + 8 * lhi);
#pragma unroll
        for (int kk = 0; kk < D / 16; kk++) asm volatile("" : "+v"(kf[kk]));   // keeps the loads ahead of the chain
#pragma unroll
        for (int kk = 0; kk < D / 16; kk++) S = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[kk], qf[kk], S, 0, 0, 0);
        return S;
    }
#pragma unroll
    for (int kk = 0; kk < D / 16; kk++) {
        const f16x8 kf = *(const f16x8 *)(sK + (32 * u + l32) * KP + 16 * kk + 8 * lhi);
        S = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[kk], S, 0, 0, 0);
    }
    return S;
}

// One row again, as the vector kernel computes it: no term of a masked cell, whatever the cache holds there; f32 probabilities.  By a whole wave,
// a lane per cell for the scores and per element for the output.
template <int D, bool PX>
__device__ __forceinline__ void exact_row(const fattn_args &a, int64_t hk, int64_t head, int64_t iq, float slope, float scale, int lane) {
    constexpr int E = (D + 63) / 64;
    const float *qp = (const float *)(a.q + iq * a.q_nb1 + head * a.q_nb2);
    const unsigned short *mrow = a.mask ? (const unsigned short *)(a.mask + iq * a.mask_nb1) : nullptr;
    const uint8_t *kh = a.k + hk * a.k_nb2, *vh = a.v + hk * a.v_nb2;
    float m = FM_NEG, l = 0.0f, acc[E];
#pragma unroll
    for (int e = 0; e < E; e++) acc[e] = 0.0f;
#pragma unroll 1
    for (int64_t c0 = 0; c0 < a.Nkv; c0 += 64) {
        const int64_t c = c0 + lane;
        const float mv = c >= a.Nkv ? -INFINITY : mrow ? half_bits_to_float(mrow[c]) : 0.0f;
        const bool valid = mv != -INFINITY;
        const uint64_t live = __ballot(valid);
        float s = FM_NEG;
        if (valid) {
            float dot = 0.0f;
#pragma unroll 1
            for (int ch = 0; ch < D / 8; ch++) {
                const f16x8 kk = *(const f16x8 *)(kh + c * a.k_nb1 + 16 * ch);
#pragma unroll
                for (int i = 0; i < 8; i++) dot = fmaf((float)(_Float16)qp[8 * ch + i], (float)kk[i], dot);
            }
            s = dot * scale;
            if (a.softcap != 0.0f) s = a.softcap * tanhf(s);
            s += slope * mv;
        }
        const float m_new = fmaxf(m, wave_max(s)), f = __expf(m - m_new), p = valid ? __expf(s - m_new) : 0.0f;
        l = l * f + wave_sum(p);
        m = m_new;
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] *= f;
#pragma unroll 1
        for (uint64_t w = live; w != 0; w &= w - 1) {
            const int j = __builtin_ctzll(w);
            const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), j));
            const _Float16 *vp = (const _Float16 *)(vh + (c0 + j) * a.v_nb1);
#pragma unroll
            for (int e = 0; e < E; e++)
                if (64 * e + lane < D) acc[e] = fmaf(pj, (float)vp[64 * e + lane], acc[e]);
        }
    }
    float *dp = a.dst + (iq * a.Hq + head) * D;
#pragma unroll
    for (int e = 0; e < E; e++)
        if (64 * e + lane < D) dp[64 * e + lane] = !PX && l == 0.0f ? 0.0f : acc[e] / l;
}

// The finished rows of a wave.  The matrix instructions multiply every cell of a tile that some query of the 32 sees, for the others by a
// probability of 0; where the cache holds something that is not finite (a cell never written, or of another sequence) that is NaN and not 0.
// Such a column cannot hide: its sum or an element is not finite.  It is computed again by exact_row, as is one whose result is rightly so.
template <int D, bool PX, int NDT>
__device__ __forceinline__ void store_rows(const fattn_args &a, const f32x16 (&o)[NDT], float l, int64_t hk, int64_t head, int64_t q0, float slope, float scale,
                                           int lane) {
    const int l32 = lane & 31, lhi = lane >> 5;
    float z = l * 0.0f;
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            if (32 * dt + 8 * (r >> 2) < D) z = fmaf(o[dt][r], 0.0f, z);
    const bool live = q0 + l32 < a.Nq;
    const uint64_t bad = __ballot(live && z != 0.0f);
    u32 again = (u32)bad | (u32)(bad >> 32);   // columns
    if (live && ((again >> l32) & 1) == 0) {
        const float sum = sum_of<PX>(l), inv = reciprocal_of<PX>(sum);
        float *dp = a.dst + ((q0 + l32) * a.Hq + head) * D;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                if (32 * dt + 8 * g >= D) continue;
                f32x4 w;
#pragma unroll
                for (int i = 0; i < 4; i++) w[i] = quotient<PX>(o[dt][4 * g + i], sum, inv);
                *(f32x4 *)(dp + 32 * dt + 8 * g + 4 * lhi) = w;
            }
    }
#pragma unroll 1
    for (; again != 0; again &= again - 1) exact_row<D, PX>(a, hk, head, q0 + __builtin_ctz(again), slope, scale, lane);   // uniform
}

// ---- prefill --------------------------------------------------------------------------------
// How far each tile of 32 queries can see: extent[t] = 1 + the last cell whose mask entry is not -inf in any of the tile's
// rows (0 when there is none).  With llama.cpp's causal mask the tiles of a prompt see a growing prefix of the cache, and the
// prefill kernel stops staging K/V tiles at that point instead of loading, scoring and then discarding them.  One group
// per tile; threads take 8 cells (16 bytes) of each row at a time.  Needs 16-byte aligned mask rows and Nkv % 8 == 0.
__global__ void __launch_bounds__(256) k_mask_extent(const uint8_t *__restrict__ mask, size_t mask_nb1, int64_t Nq, int64_t Nkv,
                                                     int32_t *__restrict__ extent) {
    __shared__ int s_max[4];
    const int64_t q0 = (int64_t)blockIdx.x * 32;
    int last = -1;
    for (int64_t c = (int64_t)threadIdx.x * 8; c < Nkv; c += 256 * 8) {
        u32x4 any = {0, 0, 0, 0};   // per 16-bit field: non-zero when some row's entry differs from -inf (0xFC00)
        for (int r = 0; r < 32; r++) {
            const int64_t iq = q0 + r < Nq ? q0 + r : Nq - 1;
            const u32x4 m = load16(mask + iq * mask_nb1 + c * 2);
#pragma unroll
            for (int i = 0; i < 4; i++) any[i] |= m[i] ^ 0xFC00FC00u;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {   // c grows, so the last assignment is the largest visible cell
            const u32 w = any[i];
            if (w & 0x0000FFFFu) last = (int)c + 2 * i;
            if (w & 0xFFFF0000u) last = (int)c + 2 * i + 1;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) last = max(last, __shfl_xor(last, off, 64));
    if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = last;
    __syncthreads();
    if (threadIdx.x == 0) extent[blockIdx.x] = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3])) + 1;
}

// Groups go to the eight XCDs round-robin by linear index and each XCD has its own L2.  Renumbered so that XCD x works through the
// x-th eighth of the grid in (head, query tile) order, the groups that read one kv head's K and V run on one XCD and find in its
// L2 what their neighbours loaded (with 8 kv heads: one head per XCD).  Query tiles are taken from the last one down: under a
// causal mask the last tile sees the most cells, and groups are started in index order, so the long groups start first and the
// short ones fill the gaps at the end (in ascending order the launch ends with the longest groups running alone: 64 slots
// and 128 tiles of 1 .. 128 half-steps finish after 96 steps instead of 64.5).  Returns the group's place (x, y) in the grid.
struct grid_pos { unsigned x, y; };
__device__ __forceinline__ grid_pos xcd_grid_pos() {
    const unsigned nx = gridDim.x;
    const uint64_t total = (uint64_t)nx * gridDim.y;
    uint64_t L = blockIdx.x + (uint64_t)nx * blockIdx.y;
    if (total % 8 == 0) L = (L % 8) * (total / 8) + L / 8;
    return grid_pos{nx - 1 - (unsigned)(L % nx), (unsigned)(L / nx)};
}

template <int D, int HPW, bool PX>
__global__ void __launch_bounds__(256, D > 128 ? 1 : 2) k_fattn_mma(fattn_args a) {
    typedef kv_stage<D, 256> stage_t;
    constexpr int QTW = 4 / HPW;   // query tiles per group
    constexpr int NDT = fm_dtiles<D>();
    __shared__ __attribute__((aligned(16))) _Float16 sK[FM_BC * stage_t::KP];
    __shared__ __attribute__((aligned(16))) _Float16 sVt[FM_BC * stage_t::VP];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, lhi = lane >> 5;
    const int groups = (int)(a.Hq / a.Hkv) / HPW;
    const grid_pos gp = xcd_grid_pos();
    const int64_t hk = gp.y / groups, hg = gp.y % groups;
    const int64_t head = (hk * groups + hg) * HPW + (wave % HPW);
    const int64_t q0 = ((int64_t)gp.x * QTW + wave / HPW) * 32;
    const int64_t iq = q0 + l32 < a.Nq ? q0 + l32 : a.Nq - 1;   // clamped: rows past Nq are computed and dropped

    f16x8 qf[D / 16];
    q_row<D> qr;
    qr.request((const float *)(a.q + iq * a.q_nb1 + head * a.q_nb2), lhi);
    float slope = alibi_slope(a, head);
    asm volatile("" : "+v"(slope));   // kept in a vector register also where the head is uniform over the group: a scalar slope makes
                                      // the compiler build a second copy of the tile loop around "slope == 1", which then spills
    const float scale = a.softcap != 0.0f ? a.scale / a.softcap : a.scale;
    const unsigned short *mrow = a.mask ? (const unsigned short *)(a.mask + iq * a.mask_nb1) : nullptr;
    const bool mask_aligned = (((uintptr_t)a.mask | a.mask_nb1) & 7) == 0;

    f32x16 o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.0f;
    float m = FM_NEG, l = 0.0f;

    // cells past kv_limit are masked for every query of this group
    int64_t kv_limit = a.Nkv;
    if (a.kv_extent) {
        int e = 0;
#pragma unroll
        for (int j = 0; j < QTW; j++) {
            const int64_t t = (int64_t)gp.x * QTW + j;
            if (t * 32 < a.Nq) e = max(e, a.kv_extent[t]);
        }
        kv_limit = e < a.Nkv ? e : a.Nkv;
    }

    stage_t st;
    u32x2 mnext[2][4];
    auto prefetch_mask = [&](int64_t kv0) {
        const bool vec_ok = mask_aligned && kv0 + FM_BC <= a.Nkv;
        fetch_mask<4>(mnext[0], mrow, vec_ok, kv0 + 4 * lhi, a.Nkv);
        fetch_mask<4>(mnext[1], mrow, vec_ok, kv0 + 32 + 4 * lhi, a.Nkv);
    };
    st.fetch(a, hk, 0, tid);   // also where the group will need no tile: behind a branch the compiler would wait for more than q
    qr.convert(qf);
    prefetch_mask(0);
    for (int64_t kv0 = 0; kv0 < kv_limit; kv0 += FM_BC) {
        __syncthreads();   // the previous tile has been consumed
        st.commit(sK, sVt, tid);
        u32x2 mcur[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int g = 0; g < 4; g++) mcur[u][g] = mnext[u][g];
        __syncthreads();
        if (kv0 + FM_BC < kv_limit) {
            st.fetch(a, hk, kv0 + FM_BC, tid);
            prefetch_mask(kv0 + FM_BC);
        }

        // scores of 64 cells for this lane's query: S[u][r] <-> cell kv0 + 32u + 8*(r/4) + 4*lhi + r%4
        f32x16 S[2];
        float mx = FM_NEG;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            S[u] = scores<D, false, PX ? fm_px_chains<D>() : 1>(qf, sK, u, l32, lhi);
            mx = max_or_nan(mx, finish_scores(S[u], mcur[u], a, scale, slope, kv0 + 32 * u, lhi, a.Nkv));
        }
        mx = half_pair_max_or_nan(mx);
        if (__ballot(!(mx <= FM_NEG)) == 0) continue;   // every cell of the tile is masked for all 32 queries (wave-uniform)
        const float m_new = lazy_max<PX>(m, mx);
        const float alpha = rescale<PX>(m, m_new);   // exactly 1 while the reference point stays
        const float m2 = exponent_of<PX>(m_new);   // finite also for a column that has seen no cell yet: exp(-inf) is 0 there too
        float rs = 0.0f;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float p = exp_rel(S[u][r], m2);
                S[u][r] = p;
                rs += p;
            }
        rs = half_pair_sum(rs);
        l = l * alpha + rs;
        m = m_new;
        if (__ballot(alpha != 1.0f) != 0) {   // wave-uniform
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
        }
        if constexpr (PX) accumulate_pv_px<D, NDT, 2>(o, S, sVt, 0, l32, lhi);
        else {
#pragma unroll
            for (int u = 0; u < 2; u++) accumulate_pv<D, NDT>(o, S[u], sVt, 0, u, l32, lhi);
        }
    }

    store_rows<D, PX, NDT>(a, o, l, hk, head, q0, slope, scale, lane);
}

// ---- prefill with few query tiles: the 32-cell parts of every K/V tile go to different waves -----------------------------------
// k_fattn_mma gives a wave 32 queries of one head and the whole 64-cell tile; a batch of a few hundred rows is then fewer groups
// than compute units, each a serial chain of tiles.  Here a group is two query heads of one kv head x the NU 32-cell parts of a
// tile of 32 NU cells: wave (hp, u) scores and accumulates cells [32u, 32u + 32) of each tile for head hp with its own soft-max
// state, and the states of a head's waves are joined pairwise through LDS at the end.  NU = 2: twice the groups of k_fattn_mma
// with half the work per wave and tile; NU = 4 (eight waves, 128-cell tiles) when even those leave one group per compute
// unit: two waves per SIMD, so that one wave's matrix instructions run under the other's soft-max arithmetic, and half the
// tile steps.
// PQ: the two columns of waves are neighbouring query tiles of one head instead of two heads (an odd number of query heads per kv head)
// SPLIT: the cells are cut into a.n_splits ranges of a.cells_per_split (whole tiles), one per group; k_fattn_half_merge joins their states
template <int D, int NU, bool PQ, bool PX, bool SPLIT = false>
__global__ void __launch_bounds__(128 * NU, NU == 2 && D <= 128 ? 2 : 1) k_fattn_mma_half(fattn_args a) {
    constexpr int NTH = 128 * NU, BC = 32 * NU;
    typedef kv_stage<D, NTH, BC> stage_t;
    constexpr int NDT = fm_dtiles<D>(), DP = 32 * NDT;
    constexpr int KV_HALVES = BC * stage_t::KP + BC * stage_t::VP;                    // f16 elements of the K tile and the V tile
    constexpr int MERGE_FLOATS = NU * (DP + 2) * 32;                                   // per (head, pair of waves): O^T [D][32], max, sum
    constexpr int SMEM_BYTES = KV_HALVES * 2 > MERGE_FLOATS * 4 ? KV_HALVES * 2 : MERGE_FLOATS * 4;
    __shared__ __attribute__((aligned(16))) uint8_t smem[SMEM_BYTES];
    _Float16 *sK = (_Float16 *)smem, *sVt = sK + BC * stage_t::KP;
    float *s_merge = (float *)smem;   // reused after the last tile

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, lhi = lane >> 5;
    const int u = wave % NU, hp = wave / NU;
    const int R = (int)(a.Hq / a.Hkv);
    const int pairs = PQ ? R : R / 2;   // heads or head pairs per kv head
    const grid_pos gp = xcd_grid_pos();
    const int64_t hk = gp.y / pairs, hg = gp.y % pairs;
    const int64_t head = PQ ? hk * pairs + hg : (hk * pairs + hg) * 2 + hp;
    const int64_t q0 = PQ ? ((int64_t)gp.x * 2 + hp) * 32 : (int64_t)gp.x * 32;
    const int64_t iq = q0 + l32 < a.Nq ? q0 + l32 : a.Nq - 1;   // clamped: rows past Nq are computed and dropped

    f16x8 qf[D / 16];
    q_row<D> qr;
    qr.request((const float *)(a.q + iq * a.q_nb1 + head * a.q_nb2), lhi);
    const float slope = alibi_slope(a, head);
    const float scale = a.softcap != 0.0f ? a.scale / a.softcap : a.scale;
    const unsigned short *mrow = a.mask ? (const unsigned short *)(a.mask + iq * a.mask_nb1) : nullptr;
    const bool mask_aligned = (((uintptr_t)a.mask | a.mask_nb1) & 7) == 0;

    f32x16 o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.0f;
    float m = FM_NEG, l = 0.0f;

    // cells past kv_limit are masked for every query of this group
    int64_t kv_limit = a.Nkv;
    if constexpr (PX) {
        if (a.kv_extent) {
            int e = a.kv_extent[PQ ? 2 * gp.x : gp.x];
            if (PQ && (int64_t)(2 * gp.x + 1) * 32 < a.Nq) e = max(e, a.kv_extent[2 * gp.x + 1]);
            kv_limit = e < a.Nkv ? e : a.Nkv;
        }
    }

    const int64_t kv_lo = SPLIT ? (int64_t)blockIdx.z * a.cells_per_split : 0;
    if (SPLIT && kv_lo + a.cells_per_split < kv_limit) kv_limit = kv_lo + a.cells_per_split;

    stage_t st;
    u32x2 mnext[4];
    auto prefetch = [&](int64_t kv0) {
        st.fetch(a, hk, kv0, tid);
        fetch_mask<4>(mnext, mrow, mask_aligned && kv0 + BC <= a.Nkv, kv0 + 32 * u + 4 * lhi, a.Nkv);
    };
    st.fetch(a, hk, kv_lo, tid);   // also where the group will need no tile: behind a branch the compiler would wait for more than q
    qr.convert(qf);
    fetch_mask<4>(mnext, mrow, mask_aligned && kv_lo + BC <= a.Nkv, kv_lo + 32 * u + 4 * lhi, a.Nkv);
    for (int64_t kv0 = kv_lo; kv0 < kv_limit; kv0 += BC) {
        __syncthreads();   // the previous tile has been consumed
        st.commit(sK, sVt, tid);
        u32x2 mcur[4];
#pragma unroll
        for (int g = 0; g < 4; g++) mcur[g] = mnext[g];
        __syncthreads();
        if (kv0 + BC < kv_limit) prefetch(kv0 + BC);
        f32x16 S1[1];
        f32x16 &S = S1[0];
        S = scores<D, (D <= 128), PX ? fm_px_chains<D>() : 1>(qf, sK, u, l32, lhi);
        float mx = finish_scores(S, mcur, a, scale, slope, kv0 + 32 * u, lhi, a.Nkv);
        mx = half_pair_max_or_nan(mx);
        if (__ballot(!(mx <= FM_NEG)) == 0) continue;   // all 32 cells masked for all 32 queries (wave-uniform; barriers are at the loop head)
        const float m_new = lazy_max<PX>(m, mx);
        const float alpha = rescale<PX>(m, m_new);   // exactly 1 while the reference point stays
        const float m2 = exponent_of<PX>(m_new);   // finite also for a column that has seen no cell yet: exp(-inf) is 0 there too
        float rs = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float p = exp_rel(S[r], m2);
            S[r] = p;
            rs += p;
        }
        rs = half_pair_sum(rs);
        l = l * alpha + rs;
        m = m_new;
        if (__ballot(alpha != 1.0f) != 0) {   // wave-uniform
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
        }
        if constexpr (PX) accumulate_pv_px<D, NDT, 1>(o, S1, sVt, u, l32, lhi);
        else accumulate_pv<D, NDT>(o, S, sVt, 0, u, l32, lhi);
    }

    // ---- the states of a head's waves are joined pairwise: u + step hands its state to u (step = 1, then 2)
#pragma unroll
    for (int step = 1; step < NU; step *= 2) {
        float *mg = s_merge + (hp * (NU / 2) + (u >> 1) / step) * (DP + 2) * 32;   // [d][query], then max, sum
        __syncthreads();
        if ((u & (2 * step - 1)) == step) {
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) mg[(32 * dt + 8 * (r >> 2) + 4 * lhi + (r & 3)) * 32 + l32] = o[dt][r];
            if (lhi == 0) {
                mg[DP * 32 + l32] = m;
                mg[(DP + 1) * 32 + l32] = l;
            }
        }
        __syncthreads();
        if ((u & (2 * step - 1)) == 0) {
            const float m1 = mg[DP * 32 + l32], l1 = mg[(DP + 1) * 32 + l32];
            const float M = fmaxf(m, m1);
            const float f0 = merge_factor<PX>(m, M), f1 = merge_factor<PX>(m1, M);
            l = l * f0 + l1 * f1;
            m = M;
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[dt][r] = o[dt][r] * f0 + mg[(32 * dt + 8 * (r >> 2) + 4 * lhi + (r & 3)) * 32 + l32] * f1;
        }
    }
    if (u != 0) return;
    if constexpr (SPLIT) {
        if (q0 + l32 >= a.Nq) return;
        const int64_t rows = a.Nq * a.Hq, at = (int64_t)blockIdx.z * rows + (q0 + l32) * a.Hq + head;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                if (32 * dt + 8 * g >= D) continue;
                f32x4 w;
#pragma unroll
                for (int i = 0; i < 4; i++) w[i] = o[dt][4 * g + i];
                *(f32x4 *)(a.ws + at * D + 32 * dt + 8 * g + 4 * lhi) = w;
            }
        if (lhi == 0) ((float2 *)(a.ws + a.n_splits * rows * D))[at] = float2{m, l};
    } else {
        store_rows<D, PX, NDT>(a, o, l, hk, head, q0, slope, scale, lane);
    }
}

// Joins the states of a row's ranges of cells, one wave per (query, head) row, in the terms of store_rows: a row that is not finite is
// computed again by exact_row.
template <int D, bool PX>
__global__ void __launch_bounds__(256) k_fattn_half_merge(fattn_args a) {
    constexpr int E = (D + 63) / 64;   // neighbouring elements of a lane (D is a multiple of E)
    typedef float part __attribute__((ext_vector_type(E == 3 ? 4 : E), aligned(4 * E)));
    static_assert(D % E == 0 && (E == 1 || E == 2 || E == 4), "elements of a lane");
    const int lane = threadIdx.x & 63;
    const int64_t rows = a.Nq * a.Hq, row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;   // whole wave
    const float2 *ml = (const float2 *)(a.ws + a.n_splits * rows * D);
    const bool live = E * lane < D;
    const float *mine_at = a.ws + row * D + (live ? E * lane : 0);   // lanes past the end repeat the first one's and are not stored
    // four ranges' values requested together, the first four ahead of the maxima; past the end the last range again, times 0
    part v[4];
    auto request = [&](int s0) {
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = *(const part *)(mine_at + (s0 + j < a.n_splits ? s0 + j : a.n_splits - 1) * (rows * D));
    };
    const float2 state = ml[(lane < a.n_splits ? lane : a.n_splits - 1) * rows + row];
    request(0);
    const float2 mine = lane < a.n_splits ? state : float2{FM_NEG, 0.0f};
    const float f = merge_factor<PX>(mine.x, wave_max_dpp(mine.x));
    const float l = wave_sum_dpp(lane < a.n_splits ? mine.y * f : 0.0f);
    part o = 0.0f;
    for (int s0 = 0;;) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float fs = s0 + j < a.n_splits ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), s0 + j)) : 0.0f;
#pragma unroll
            for (int e = 0; e < E; e++) o[e] = fmaf(v[j][e], fs, o[e]);
        }
        s0 += 4;
        if (s0 >= a.n_splits) break;   // uniform
        request(s0);
    }
    float z = l * 0.0f;
#pragma unroll
    for (int e = 0; e < E; e++) z = fmaf(o[e], 0.0f, z);
    const int64_t iq = row / a.Hq, head = row % a.Hq;
    if (__ballot(z != 0.0f) != 0) {
        exact_row<D, PX>(a, head / (a.Hq / a.Hkv), head, iq, alibi_slope(a, head), a.softcap != 0.0f ? a.scale / a.softcap : a.scale, lane);
        return;
    }
    const float sum = sum_of<PX>(l), inv = reciprocal_of<PX>(sum);
    if (live) {
#pragma unroll
        for (int e = 0; e < E; e++) a.dst[row * D + E * lane + e] = quotient<PX>(o[e], sum, inv);
    }
}

// How many ranges the cells are cut into.  A group's walk is a serial chain, so a launch of few groups takes as long as one of them however idle
// the chip is; the states of more ranges cost a merge launch and their way through memory.  The time in us of n ranges, from a sweep over
// (64 .. 256 head size, 24 .. 256 groups, 2 .. 256 tiles of 64 cells, n = 1 .. 16), which it meets within some 15 %: a tile step takes
// 0.95 (D 64), 1.4 (up to 128) or 3.4 us (256: one group per compute unit), 1.34 times that with a second group on the compute unit; the merge 4
// and 8 bytes per value and range at 4 TB/s.  Before / after, us: 64 rows over 8192 cells, 32 / 8 heads, D 128 146 -> 32; 343 x 3840, 4 / 4 heads, D 64
// 51 -> 18; 268 x 3776, 32 / 8, D 128 77 -> 50; 512 x 4096 79.8 -> 69.2 (n = 2); 300 x 2500, 8 / 8, D 256 136 -> 41; not cut: 560 x 672, 16 / 4 (22.5; 27 in three).
// Probabilities of f32 precision: one launch up to 2048 cells.  Shorter walks gain too, but over few cells the sum of ranges is in places further from 64 bits
// than one walk; whole / in ranges, us and error: 300 rows x 512 cells, 8 / 8 heads, D 256 36.5 / 26.7 and 1.74e-7 / 1.76e-7, D 80 16.6 / 13.6 and 1.64e-7 /
// 1.68e-7, x 1024 26.0 / 16.2 and 1.75e-7 / 1.77e-7.  At 2048 cells the errors are smaller in ranges (300 rows, D 256 109.8 / 39.5 us, 2.21e-7 / 2.02e-7;
// 64 rows, 32 / 8 heads, D 80 43.6 / 16.7, 2.00e-7 / 1.97e-7; 512 rows are not cut): the line could lie there, it has not been looked for between 1024 and 2048.
static bool half_may_split(const fattn_args &a, bool px) { return (!px || a.Nkv > 2048) && a.ws != nullptr && ((uintptr_t)a.ws & 15) == 0; }
static int64_t plan_half(int64_t D, int64_t groups, int64_t rows, int64_t tiles, bool wide, size_t ws_bytes) {
    const float step = D == 64 ? 0.95f : D <= 128 ? 1.4f : 3.4f;
    int64_t best = 1;
    float best_us = 0.0f, whole = 0.0f;
    for (int64_t n = 1; n <= 64 && n <= tiles; n++) {
        if (n > 1 && ws_bytes < (size_t)n * (size_t)rows * (size_t)(D + 2) * sizeof(float)) break;
        const int64_t g = groups * n, slots = D <= 128 ? 512 : 256;
        const float busy = g <= 256 ? 1.0f : (float)((g + slots - 1) / slots) * (D <= 128 ? 1.34f : 1.0f);
        float us = (float)((tiles + n - 1) / n) * step * busy;
        if (n == 1 && wide) us *= 0.9f;   // eight waves on 128-cell tiles
        if (n > 1) us += 4.0f + (float)(rows * n * D) * 8.0f / 4e6f;
        if (n == 1) whole = us;
        if (n == 1 || (us < best_us && us < 0.9f * whole)) {
            best = n;
            best_us = us;
        }
    }
    return best;
}

template <int D, bool PQ, bool PX>
int launch_half(hipStream_t s, fattn_args a, size_t ws_bytes) {
    const int64_t R = a.Hq / a.Hkv, n_tiles = (a.Nq + 31) / 32;
    dim3 grid((unsigned)(PQ ? (n_tiles + 1) / 2 : n_tiles), (unsigned)(a.Hkv * (PQ ? R : R / 2)));
    const int64_t groups = (int64_t)grid.x * grid.y, rows = a.Nq * a.Hq, tiles = (a.Nkv + 63) / 64;
    // at most one group per compute unit and a long cache: eight waves on 128-cell tiles (an earlier form of the kernel, 512 rows: 4096 cells 112 -> 103 us).
    // Below 1024 cells four waves are quicker, four / eight, us: 512 rows, D 128, 32 / 8 heads, 512 cells 17.3 / 19.3, 768 22.2 / 23.3; D 80, 32 / 32, 512 17.5 / 18.5,
    // 960 27.1 / 31.0; D 112, 32 / 8, 960 33.5 / 37.1; quantized output, D 64, 512 19.2 / 19.4.  Head size 256: the eight waves' registers do not fit.
    const bool wide = D <= 128 && groups <= 256 && a.Nkv >= 1024;
    // the groups read the mask extents, at the front of the scratch memory, while others write their states: those lie behind
    if (a.kv_extent) {
        const size_t used = ((size_t)((a.Nq + 31) / 32) * sizeof(int32_t) + 15) & ~(size_t)15;
        a.ws += used / sizeof(float);
        ws_bytes = ws_bytes > used ? ws_bytes - used : 0;
    }
    const int64_t n = half_may_split(a, PX) ? plan_half(D, groups, rows, tiles, wide, ws_bytes) : 1;
    a.cells_per_split = (tiles + n - 1) / n * 64;
    a.n_splits = (int)((a.Nkv + a.cells_per_split - 1) / a.cells_per_split);   // no empty range
    grid.z = (unsigned)a.n_splits;
    if constexpr (D <= 128) {
        if (wide && a.n_splits == 1) {
            MI355_LAUNCH((k_fattn_mma_half<D, 4, PQ, PX>), grid, dim3(512), 0, s, a);
            return launch_status("k_fattn_mma_half");
        }
    }
    if (a.n_splits == 1) {
        MI355_LAUNCH((k_fattn_mma_half<D, 2, PQ, PX>), grid, dim3(256), 0, s, a);
        return launch_status("k_fattn_mma_half");
    }
    MI355_LAUNCH((k_fattn_mma_half<D, 2, PQ, PX, true>), grid, dim3(256), 0, s, a);
    const int rc = launch_status("k_fattn_mma_half");
    if (rc != MI355_OK) return rc;
    MI355_LAUNCH((k_fattn_half_merge<D, PX>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, a);
    return launch_status("k_fattn_half_merge");
}

template <int D, int HPW, bool PX>
int launch(hipStream_t s, const fattn_args &a) {
    constexpr int QTW = 4 / HPW;
    const int64_t groups = (a.Hq / a.Hkv) / HPW;
    const dim3 grid((unsigned)((a.Nq + 32 * QTW - 1) / (32 * QTW)), (unsigned)(a.Hkv * groups));
    MI355_LAUNCH((k_fattn_mma<D, HPW, PX>), grid, dim3(256), 0, s, a);
    return launch_status("k_fattn_mma");
}

template <int D, bool PX>
int launch_hpw(hipStream_t s, const fattn_args &a) {
    const int64_t R = a.Hq / a.Hkv;
    if (R % 4 == 0) return launch<D, 4, PX>(s, a);
    if (R % 2 == 0) return launch<D, 2, PX>(s, a);
    return launch<D, 1, PX>(s, a);
}

// Pairs of probabilities: head sizes 112 and 128 always in halves (the registers of whole tiles do not fit: 50 and 33 spills; 2048 x 2048 cells,
// 32 / 8 heads: 165 -> 139 and 160 -> 155 us), head size 64 too (the error of its longer sums would exceed the vector kernel's, 1.39e-7 against 1.36e-7; halves 1.34e-7)
template <int D, bool PX>
int launch_head(hipStream_t s, const fattn_args &a, size_t ws_bytes, bool pq, bool half) {
    constexpr bool HALVES_ONLY = PX && (D == 64 || D == 112 || D == 128);
    if constexpr (!HALVES_ONLY) {
        if (!half) return launch_hpw<D, PX>(s, a);
    }
    return pq ? launch_half<D, true, PX>(s, a, ws_bytes) : launch_half<D, false, PX>(s, a, ws_bytes);
}

// ---- decode / small batches: the 32 MFMA columns are (token, head of the GQA group) pairs -------
// A 256-thread group owns one kv head, NT = 32 / R tokens and one kv split, so the K/V bytes of
// a kv head are read once for all R query heads.  Its four waves are (u, h): u picks the 32-cell
// half of each 64-cell tile the wave scores, h the half of the head dimension it accumulates.
// States are merged through LDS; a split writes (O, max, sum) partials for k_fattn_combine.
template <int D>
__global__ void __launch_bounds__(256, 2) k_fattn_mma_dec(fattn_args a, int R, int NT) {
    typedef kv_stage<D, 256> stage_t;
    constexpr int NDT = D / 64;   // 32-row O^T tiles per wave
    __shared__ __attribute__((aligned(16))) _Float16 sK[FM_BC * stage_t::KP];
    __shared__ __attribute__((aligned(16))) _Float16 sVt[FM_BC * stage_t::VP];
    float *s_merge = (float *)sK;   // reused after the last tile: per h, [D/2 + 2][32] floats of the u = 1 wave
    static_assert(sizeof(_Float16) * FM_BC * stage_t::KP >= sizeof(float) * (D + 4) * 32, "merge buffer does not fit the K tile");

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, lhi = lane >> 5;
    const int u = wave & 1, h = wave >> 1;
    const int split = blockIdx.x;
    const int64_t hk = blockIdx.y;
    const int col_tok = l32 / R, col_head = l32 % R;
    const bool col_live = col_tok < NT && (int64_t)blockIdx.z * NT + col_tok < a.Nq;
    const int64_t iq = col_live ? (int64_t)blockIdx.z * NT + col_tok : a.Nq - 1;
    const int64_t head = hk * R + (col_live ? col_head : 0);

    f16x8 qf[D / 16];
    q_row<D> qr;
    qr.request((const float *)(a.q + iq * a.q_nb1 + head * a.q_nb2), lhi);
    const float slope = alibi_slope(a, head);
    const float scale = a.softcap != 0.0f ? a.scale / a.softcap : a.scale;
    const unsigned short *mrow = a.mask ? (const unsigned short *)(a.mask + iq * a.mask_nb1) : nullptr;
    const bool mask_aligned = (((uintptr_t)a.mask | a.mask_nb1) & 7) == 0;

    f32x16 o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.0f;
    float m = FM_NEG, l = 0.0f;

    const int64_t c_begin = (int64_t)split * a.cells_per_split;
    const int64_t c_end = c_begin + a.cells_per_split < a.Nkv ? c_begin + a.cells_per_split : a.Nkv;

    // two tiles of K/V (and their mask entries) are always in flight: tile i + 2 is requested as soon as the
    // registers of tile i have been written to LDS
    stage_t st0, st1;
    u32x2 mn0[4], mn1[4];
    auto prefetch = [&](stage_t &st, u32x2 (&mn)[4], int64_t kv0) {
        st.fetch(a, hk, kv0, tid);
        fetch_mask<4>(mn, mrow, mask_aligned && kv0 + FM_BC <= a.Nkv, kv0 + 32 * u + 4 * lhi, a.Nkv);
    };
    auto tile = [&](stage_t &st, u32x2 (&mn)[4], int64_t kv0) {
        __syncthreads();   // the previous tile has been consumed
        st.commit(sK, sVt, tid);
        u32x2 mcur[4];
#pragma unroll
        for (int g = 0; g < 4; g++) mcur[g] = mn[g];
        __syncthreads();
        if (kv0 + 2 * FM_BC < c_end) prefetch(st, mn, kv0 + 2 * FM_BC);
        f32x16 S = scores<D>(qf, sK, u, l32, lhi);
        float mx = finish_scores_dec(S, mcur, a, scale, slope, kv0 + 32 * u, lhi, c_end);
        mx = half_pair_max(mx);
        if (__ballot(mx > FM_NEG) == 0) return;   // all 32 cells masked for every column (wave-uniform)
        const float m_new = fmaxf(m, mx);
        const float alpha = __expf(m - m_new);
        float rs = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float p = S[r] > FM_NEG ? __expf(S[r] - m_new) : 0.0f;
            S[r] = p;
            rs += p;
        }
        rs = half_pair_sum(rs);
        l = l * alpha + rs;
        m = m_new;
        if (__ballot(alpha != 1.0f) != 0) {   // wave-uniform: most tiles do not raise any column's maximum
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
        }
        accumulate_pv<D, NDT>(o, S, sVt, h * NDT, u, l32, lhi);
    };
    st0.fetch(a, hk, c_begin, tid);   // (no range of cells is empty)
    qr.convert(qf);
    fetch_mask<4>(mn0, mrow, mask_aligned && c_begin + FM_BC <= a.Nkv, c_begin + 32 * u + 4 * lhi, a.Nkv);
    if (c_begin + FM_BC < c_end) prefetch(st1, mn1, c_begin + FM_BC);
    for (int64_t kv0 = c_begin; kv0 < c_end; kv0 += 2 * FM_BC) {
        tile(st0, mn0, kv0);
        if (kv0 + FM_BC < c_end) tile(st1, mn1, kv0 + FM_BC);   // uniform over the group
    }

    // ---- merge the u = 1 wave into the u = 0 wave of the same h
    float *mg = s_merge + h * (D / 2 + 2) * 32;   // [d_local][col], then max, sum
    __syncthreads();
    if (u == 1) {
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) mg[(32 * dt + 8 * (r >> 2) + 4 * lhi + (r & 3)) * 32 + l32] = o[dt][r];
        if (lhi == 0) {
            mg[(D / 2) * 32 + l32] = m;
            mg[(D / 2 + 1) * 32 + l32] = l;
        }
    }
    __syncthreads();
    if (u != 0 || !col_live) return;
    {
        const float m1 = mg[(D / 2) * 32 + l32], l1 = mg[(D / 2 + 1) * 32 + l32];
        const float M = fmaxf(m, m1);
        const float f0 = __expf(m - M), f1 = __expf(m1 - M);
        l = l * f0 + l1 * f1;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[dt][r] = o[dt][r] * f0 + mg[(32 * dt + 8 * (r >> 2) + 4 * lhi + (r & 3)) * 32 + l32] * f1;
        m = M;
    }
    const int d_first = h * (D / 2);   // this wave's slice of the head
    if (a.n_splits == 1) {
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        float *dp = a.dst + (iq * a.Hq + head) * D + d_first;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) {
            float w[16];
            float amax = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                w[r] = o[dt][r] * inv;
                amax = fmaxf(amax, fabsf(w[r]));
            }
#pragma unroll
            for (int g = 0; g < 4; g++) *(f32x4 *)(dp + 32 * dt + 8 * g + 4 * lhi) = f32x4{w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]};
            if (a.act_q) {   // Q8_1 of this 32-element block of the head (quantize_row_q8_1_ref, ggml-quants.c:220-253)
                amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
                float d, id;
                q8_scale(amax, d, id);
                int sum = 0;
                const int64_t e0 = head * D + d_first + 32 * dt;   // first element of the block inside the activation row
                int8_t *qrow = a.act_q + iq * a.Hq * D + e0;
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    u32 packed = 0;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int q = q8_level(w[4 * g + i], id);
                        sum += q;
                        packed |= (u32)(q & 0xFF) << (8 * i);
                    }
                    *(u32 *)(qrow + 8 * g + 4 * lhi) = packed;
                }
                sum += __shfl_xor(sum, 32, 64);
                if (lhi == 0) {
                    act_ds e;
                    e.d = half_bits_to_float(float_to_half_bits(d));
                    e.sum = sum;
                    a.act_s[iq * (a.Hq * D / 32) + e0 / 32] = e;
                }
            }
        }
    } else {
        float *p = a.ws + ((iq * a.Hq + head) * a.n_splits + split) * (D + 2);
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int i = 0; i < 4; i++) p[d_first + 32 * dt + 8 * g + 4 * lhi + i] = o[dt][4 * g + i];
        if (h == 0 && lhi == 0) {
            p[D] = m;
            p[D + 1] = l;
        }
    }
}

template <int D>
int launch_dec(hipStream_t s, const fattn_args &a) {
    const int R = (int)(a.Hq / a.Hkv);
    const int NT = 32 / R;
    const dim3 grid((unsigned)a.n_splits, (unsigned)a.Hkv, (unsigned)((a.Nq + NT - 1) / NT));
    MI355_LAUNCH(k_fattn_mma_dec<D>, grid, dim3(256), 0, s, a, R, NT);
    return launch_status("k_fattn_mma_dec");
}

}  // namespace

// From how many (query, head) pairs on the matrix-core kernels are ahead of the vector kernel, which splits the cells over groups and so
// fills the chip with any number of pairs, while a tile of 32 queries walks all cells in one serial chain (1.1 us per 64 cells of D 80).
// Smallest sizes at which no call of the grid {4 .. 64 heads} x {16 .. 384 rows} x {64 .. 16384 cells} x head sizes was slower: us, vector / matrix,
// 16384 cells: D 80, 4 heads, 16 rows 35 / 291; D 256, 8 heads, 64 rows 318 / 818; D 64, 16 heads, 64 rows 146 / 253, 96 rows 232 / 252;
// D 80, 32 heads, 48 rows 465 / 295; 64 cells, D 256, 32 heads, 48 rows 11 / 15, 64 rows 13.6 / 15.2.
static int64_t px_min_pairs(int64_t D, int64_t Nkv) { return Nkv < 512 ? 2049 : D == 64 ? 1537 : 1152; }

int launch_fattn_mma(hipStream_t s, fattn_args &a, int64_t D, size_t ws_bytes) {
    if (a.Hkv * (a.Hq / a.Hkv) > 65535 || (a.Nq + 31) / 32 > 0x7fffffff) return 1;
    if ((a.q_nb1 % 16) != 0 || (a.q_nb2 % 16) != 0) return 1;
    if (a.k_nb1 >= (size_t(1) << 24) || a.v_nb1 >= (size_t(1) << 24)) return 1;   // kv_stage: a tile's rows within 32-bit offsets
    // head sizes 64 and 128: f16 probabilities, except where the output is also quantized
    const bool px = a.act_q != nullptr || (D != 64 && D != 128);
    if (px && a.Nq * a.Hq < px_min_pairs(D, a.Nkv)) return 1;
    a.kv_extent = nullptr;
    const int64_t n_tiles = (a.Nq + 31) / 32;
    // The pre-pass pays when there are more groups than the chip holds at once (two per compute unit): then a group that stops
    // early makes room for the next one.  With fewer groups the launch takes as long as its longest group either way.
    const int64_t n_groups = n_tiles * a.Hq / 4;
    if (n_groups > 512 && a.mask && a.ws && ws_bytes >= (size_t)n_tiles * sizeof(int32_t) && (((uintptr_t)a.mask | a.mask_nb1) & 15) == 0 &&
        a.Nkv % 8 == 0 && a.Nkv >= 2 * FM_BC && a.Nkv < 0x7fffffff) {
        MI355_LAUNCH(k_mask_extent, dim3((unsigned)n_tiles), dim3(256), 0, s, a.mask, a.mask_nb1, a.Nq, a.Nkv, (int32_t *)a.ws);
        const int rc = launch_status("k_mask_extent");
        if (rc != MI355_OK) return rc;
        a.kv_extent = (const int32_t *)a.ws;
    }
    // few query tiles (a batch of a few hundred rows): twice the groups with half a K/V tile per wave, while the chip is not full
    const int64_t R = a.Hq / a.Hkv;
    // (an odd number of query heads per kv head pairs neighbouring query tiles: 512 rows over 1024 cells, 32 heads, D 128: 40 -> 31 us).
    // Against the vector kernel, which served the other head sizes and the quantized output before (us; error against 64-bit arithmetic on the
    // same operands; f16 probabilities would be 1.5e-4 .. 2.1e-4): 512 x 512 cells, 32 / 32 heads, D 80: 203 -> 18.3, 1.28e-7 -> 1.25e-7;
    // 2048 x 2048, 32 / 8 heads: D 80 2046 -> 111, 1.56e-7 -> 1.49e-7; D 112 2049 -> 139, 1.55e-7 -> 1.47e-7; D 256 4346 -> 252, 1.71e-7 -> 1.59e-7;
    // D 128 with quantized output 2056 -> 155, 1.55e-7 -> 1.44e-7, 768 x 2048 812 -> 91, 2.49e-7 -> 2.05e-7.
    const bool pq = R % 2 != 0, half = (pq ? (n_tiles + 1) / 2 * a.Hq : n_tiles * a.Hq / 2) <= 512;
#define MI355_FM_HEAD(D_, PX_) return launch_head<D_, PX_>(s, a, ws_bytes, pq, half);
    switch (D) {
        case 64: if (px) MI355_FM_HEAD(64, true) else MI355_FM_HEAD(64, false)
        case 80: MI355_FM_HEAD(80, true)
        case 96: MI355_FM_HEAD(96, true)
        case 112: MI355_FM_HEAD(112, true)
        case 128: if (px) MI355_FM_HEAD(128, true) else MI355_FM_HEAD(128, false)
        case 256: MI355_FM_HEAD(256, true)
        default: return 1;
    }
#undef MI355_FM_HEAD
}

// Few query rows: returns 1 when the shape is not served.  a.n_splits / a.cells_per_split (a multiple of 64) are set by the caller.
int launch_fattn_mma_dec(hipStream_t s, fattn_args &a, int64_t D) {
    const int64_t R = a.Hq / a.Hkv;
    if (R > 32 || a.Hkv > 65535 || (a.q_nb1 % 16) != 0 || (a.q_nb2 % 16) != 0 || a.cells_per_split % FM_BC != 0) return 1;
    if ((a.Nq + (32 / R) - 1) / (32 / R) > 65535) return 1;
    if (a.k_nb1 >= (size_t(1) << 24) || a.v_nb1 >= (size_t(1) << 24)) return 1;   // kv_stage: a tile's rows within 32-bit offsets
    switch (D) {
        case 64: return launch_dec<64>(s, a);
        case 128: return launch_dec<128>(s, a);
        default: return 1;
    }
}

}  // namespace mi355
