// The body of the GEMV launches (gemv.hip, gemv_qkv.hip): rows of one matrix against one to eight quantized activation rows.
#pragma once
#include "common.hpp"
#include "kv_blocks.hpp"
#include "qdot.hpp"
#include "norm_quant.hpp"

namespace mi355 {

struct gemv_item {
    const uint8_t *W;
    float *dst;
    const float *residual;   // may be null; same shape/stride as dst; may alias dst
    int64_t N;
    int64_t dst_stride;
    int type;
    int first_group;         // index of this matrix's first group in the launch
    int epi;                 // EPI_*: what happens to a finished row
    int64_t nb1, nb2;        // EPI_*_CACHE: byte strides of a cache cell and of a head inside it (dst = cache base)
                             // EPI_*_QCACHE: block index of cell 0 within the tensor that owns the cache memory (dst = its data) and
                             // that tensor's blocks per row in the device row layout (0: plain ggml blocks)
    int ctype;               // EPI_*_QCACHE: MI355_Q8_0 or MI355_Q4_0
};
enum { EPI_STORE = 0, EPI_ROPE = 1, EPI_ROPE_CACHE = 2, EPI_CACHE = 3, EPI_ROPE_QCACHE = 4, EPI_QCACHE = 5 };

// rotary embedding of the Q/K rows produced by the fused QKV launch (mode 0: adjacent pairs)
struct gemv_rope {
    const int32_t *pos;      // [B] rope position of each activation row
    const int32_t *cells;    // [B] cache cell of each activation row
    const float *ff;         // frequency factors [n_dims/2] or null
    int D, n_dims;
    float theta_scale, freq_scale, ext_factor, attn_factor, corr0, corr1;
    const float2 *table;     // k_gemv_qkv_norm<true>: {cos, sin} of every pair of the one activation row from k_rope_table; the other launches work out their own (same bits)
    const float *nx, *nw;    // the launches with the norm: the f32 row to normalise and the norm weights (the group quantizes it into its LDS copy itself)
    float neps;
};

// rope_yarn, same roundings as k_rope (glue.hip) and k_rope_kv_store (fused.hip); ggml-cpu.c:9268-9306
__device__ __forceinline__ void rope_coeffs(const gemv_rope &a, int pos, int pair, float &c, float &s) {
    const float theta_extrap = (float)pos * powf(a.theta_scale, (float)pair) / (a.ff ? a.ff[pair] : 1.0f);
    const float theta_interp = a.freq_scale * theta_extrap;
    float theta = theta_interp, mscale = a.attn_factor;
    if (a.ext_factor != 0.0f) {
        const float yv = ((float)pair - a.corr0) / fmaxf(0.001f, a.corr1 - a.corr0);
        const float ramp = (1.0f - fminf(1.0f, fmaxf(0.0f, yv))) * a.ext_factor;
        theta = theta_interp * (1.0f - ramp) + theta_extrap * ramp;
        mscale *= 1.0f + 0.1f * logf(1.0f / a.freq_scale);
    }
    c = cosf(theta) * mscale;
    s = sinf(theta) * mscale;
}
__device__ __forceinline__ void rope_apply(float c, float s, float x0, float x1, float &y0, float &y1) {
    y0 = sub_rn(mul_rn(x0, c), mul_rn(x1, s));
    y1 = add_rn(mul_rn(x0, s), mul_rn(x1, c));
}
struct gemv_batch {
    gemv_item it[4];
    int n;
};

// COH: results are stored with device scope (written through to where every XCD sees them), for launches whose last
// group reads rows produced by other groups
// LDSA: the group copies the quantized activation (NCOLS rows of K levels, then their scales) into s_act once and its four
// waves read it from there; otherwise every wave reads it from memory.  On the 14336 x 4096 Q4_K product the activation
// reads of the 7168 waves (36 MB from L2) outweighed the 33 MB of weights and competed with them: 8.7 -> 7.9 us with the
// copy in LDS.  The copy is requested ahead of the first step's weights: loads return in the order of their issue.
template <int TYPE, int NCOLS, int RPW, bool QKV = false, bool COH = false, bool LDSA = false>
__device__ __forceinline__ void gemv_body(const gemv_item &m, int group, const int8_t *__restrict__ aq,
                                          const act_ds *__restrict__ ads, int K, const gemv_rope *rp = nullptr, uint8_t *s_act = nullptr) {
    typedef wq<TYPE> T;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = ((int64_t)group * 4 + wave) * RPW;
    const bool wave_live = row0 < m.N;   // uniform over the wave
    if (!LDSA && !wave_live) return;     // with the copy in LDS a wave without rows still takes its share of the copy

    const row_layout L = make_row_layout(TYPE, K);
    const int nchunks = K / T::CHUNK;
    const int nblk = K >> 5;   // Q8_1 blocks per activation row

    const uint8_t *rows[RPW];
#pragma unroll
    for (int r = 0; r < RPW; r++) {
        const int64_t row = row0 + r < m.N ? row0 + r : m.N - 1;   // clamp: tail rows recompute the last row, never stored
        rows[r] = m.W + row * L.row_bytes;
    }

    float acc[RPW][NCOLS];
#pragma unroll
    for (int r = 0; r < RPW; r++)
#pragma unroll
        for (int c = 0; c < NCOLS; c++) acc[r][c] = 0.0f;

    // The order of the requests: a wave's loads return as they were issued, so the activation comes first (with what the QKV epilogue needs to know), the first step's
    // weights behind it, and what can be computed without the weights is done while they are on their way.
    // Without the copy the Q/K/V launch requests the first step's weights ahead of the rotations too: of three and four tokens, of Q8_0, and of two tokens of the types whose chunks are the
    // widest.  us, 32 / 8 heads, 4096 elements, weights behind the rotations / ahead: four tokens Q6_K 11.8 / 10.3, Q4_K with Q6_K for V 10.1 / 9.1, Q8_0 10.2 / 9.5, three Q4_K 8.8 / 7.4,
    // one Q8_0 7.9 / 7.6, two Q4_K 7.4 / 6.7; but one of Q4_0 6.0 / 6.1, of Q4_K with Q6_K for V 6.6 / 7.0, two of Q6_K 8.1 / 8.7.
    constexpr bool AHEAD = QKV && !LDSA && (NCOLS >= 3 || TYPE == MI355_Q8_0 || (T::CHUNK == 64 && NCOLS == 2));
    typename T::chunk w_first[RPW];
    float rope_c = 1.0f, rope_s = 0.0f;
    int pos = 0, cell = 0;
    if constexpr (QKV) {
        const int col = lane < NCOLS ? lane : NCOLS - 1;
        if (rp->pos) pos = rp->pos[col];       // null where no matrix of the launch is rotated
        if (rp->cells) cell = rp->cells[col];  // ... or goes to a cache
    }
    // QKV: lane c finishes activation row c.  Its rotation depends on nothing the product computes (the empty asm keeps it from being moved behind the loop, next
    // to its use).
    auto rotation = [&]() {
        if (lane < NCOLS) {
            const gemv_rope &R = *rp;
            const int d = (int)(row0 % R.D);
            if ((m.epi == EPI_ROPE || m.epi == EPI_ROPE_CACHE) && d < R.n_dims) rope_coeffs(R, pos, d >> 1, rope_c, rope_s);
        }
        asm volatile("" : "+v"(rope_c), "+v"(rope_s));
    };
    const int c_first = lane < nchunks ? lane : nchunks - 1;
    if constexpr (LDSA) {
        act_copy<NCOLS, 256> copy;
        copy.request(aq, ads, K);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RPW; r++) w_first[r] = T::load_w(rows[r], L, c_first);
        if constexpr (QKV) rotation();
        copy.commit(s_act, aq, ads, K);
        __syncthreads();
        if (!wave_live) return;
        aq = (const int8_t *)s_act;
        ads = (const act_ds *)(s_act + NCOLS * K);
    } else if constexpr (QKV) {
        if constexpr (AHEAD) {
#pragma unroll
            for (int r = 0; r < RPW; r++) w_first[r] = T::load_w(rows[r], L, c_first);
            __builtin_amdgcn_sched_barrier(0);
        }
        rotation();
    }

    for (int c0 = 0; c0 < nchunks; c0 += 64) {
        const int c = c0 + lane;
        if (c < nchunks) {
            typename T::chunk w[RPW];
#pragma unroll
            for (int r = 0; r < RPW; r++) {
                if ((LDSA || AHEAD) && c0 == 0) w[r] = w_first[r];
                else w[r] = T::load_w(rows[r], L, c);
            }
#pragma unroll
            for (int col = 0; col < NCOLS; col++) {
                const typename T::act A = T::load_a(aq + (int64_t)col * K, ads + col * nblk, c);
#pragma unroll
                for (int r = 0; r < RPW; r++) {
                    const chunk_dots d = T::dots(w[r], A);
                    acc[r][col] = T::accumulate(acc[r][col], w[r], A, d);
                }
            }
        }
    }

    if constexpr (QKV) {
        // RPW == 2: the wave owns the adjacent rows (row0, row0 + 1) = one rotation pair of one head.
        // Every lane gets all sums; lane c finishes activation row c.
        static_assert(RPW == 2, "the rope epilogue pairs the two rows of a wave");
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int c = 0; c < NCOLS; c++) {
            const float a0 = wave_sum_dpp(acc[0][c]), a1 = wave_sum_dpp(acc[1][c]);
            if (lane == c) { s0 = a0; s1 = a1; }
        }
        if (lane < NCOLS && row0 + 1 < m.N) {
            const gemv_rope &R = *rp;
            const int64_t head = row0 / R.D;
            const int d = (int)(row0 % R.D);
            float y0 = s0, y1 = s1;
            if ((m.epi == EPI_ROPE || m.epi == EPI_ROPE_CACHE) && d < R.n_dims) rope_apply(rope_c, rope_s, s0, s1, y0, y1);
            if (m.epi == EPI_ROPE || m.epi == EPI_STORE) {
                float *o = m.dst + lane * m.dst_stride + row0;
                o[0] = y0;
                o[1] = y1;
            } else {
                _Float16 *o = (_Float16 *)((uint8_t *)m.dst + (int64_t)cell * m.nb1 + head * m.nb2) + d;
                o[0] = (_Float16)y0;
                o[1] = (_Float16)y1;
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < RPW; r++)
#pragma unroll
            for (int c = 0; c < NCOLS; c++) {
                const float s = wave_sum_dpp(acc[r][c]);
                if (lane == 0 && row0 + r < m.N) {
                    const int64_t o = c * m.dst_stride + row0 + r;
                    const float v = m.residual ? s + m.residual[o] : s;
                    if constexpr (COH) __hip_atomic_store(m.dst + o, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    else m.dst[o] = v;
                }
            }
    }
}

// The Q/K/V launch when K and / or V go to a Q8_0 / Q4_0 cache: groups of EIGHT waves.  QUANT: the group's 32 rows (four per wave)
// are one block of a cache row; the finished, rotated values meet in LDS and wave c quantizes the block of activation row c
// (quantize_row_q8_0_ref / quantize_row_q4_0_ref, as the cache copies of kv_quant.hip do); m.N is a multiple of 32, so every wave is
// live.  !QUANT: 16 rows per group (two per wave) with the epilogues of gemv_body.  Every row sum is formed exactly as in gemv_body.
// (Groups of four waves that took their eight rows each in two passes of four were measured first: 14.6 us against 10.3 us for the
// launch with f16 stores on the Llama-8B shapes - the groups of 32 rows ran twice as long as the others.)
template <int TYPE, int NCOLS, bool NORM, bool QUANT>
__device__ __forceinline__ void gemv_body_qc(const gemv_item &m, int group, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int K,
                                             const gemv_rope &R, uint8_t *s_act) {
    typedef wq<TYPE> T;
    constexpr int NW = 8, RPW = QUANT ? 4 : 2, NP = RPW / 2;
    static_assert(!NORM || NCOLS == 1, "the norm is one row's");
    static_assert(NCOLS <= 4, "wave c quantizes activation row c");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = ((int64_t)group * NW + wave) * RPW;
    const bool wave_live = row0 < m.N;   // uniform over the wave; always true with QUANT
    if (!NORM && !wave_live) return;     // with NORM a wave without rows still takes its share of the norm and its barriers
    const row_layout L = make_row_layout(TYPE, K);
    const int nchunks = K / T::CHUNK;
    const int nblk = K >> 5;

    const uint8_t *rows[RPW];
#pragma unroll
    for (int r = 0; r < RPW; r++) {
        const int64_t row = row0 + r < m.N ? row0 + r : m.N - 1;   // clamp: tail rows recompute the last row, never stored
        rows[r] = m.W + row * L.row_bytes;
    }

    // NORM.  Types whose row is two steps of 64 chunks: the row first, the weights behind it - a wave's loads return in the order of their issue - and the rotations worked out while both
    // are on their way.  The second step of four rows per wave is requested when the registers of the normalised row are free; of the K-quants, whose chunks are the largest, it waits for
    // the first one's.  Types of one step: rotations, weights, row.  8B shapes in a chain of launches, Q8_0 caches, us, every type's own matrices: the row behind the weights and the second
    // step behind the sums of the first / this (the same before loads of the row were without branches): Q8_0 12.3 / 11.2 (11.7), Q4_0 9.2 / 8.5 (9.5), Q6_K 12.1 / 11.4 (12.3), Q5_K 13.2 / 11.9
    // (13.7), IQ4_XS 10.9 / 10.4 (11.4), Q4_K 10.1 / 10.1 (10.7).  The row first for types of one step: Q5_K 13.5, Q4_K 10.0; both steps of four rows ahead: spills, Q6_K for V 14.1.
    typedef late_chunk<TYPE> G;
    constexpr int STEPS = 64 / T::CHUNK;   // steps of 64 chunks in a row of 4096
    constexpr int FIRST = QUANT ? 1 : STEPS;
    typename G::raw wn[STEPS][RPW];
    auto request = [&](int from, int to) {
#pragma unroll
        for (int p = 0; p < STEPS; p++)
#pragma unroll
            for (int r = 0; r < RPW; r++) {
                const int c = p * 64 + lane;
                if (p >= from && p < to) wn[p][r] = G::load(rows[r], L, c < nchunks ? c : nchunks - 1);
            }
    };
    norm_row<NW> row;
    __shared__ float s_norm[4];
    int pos = 0, cell = 0;
    if constexpr (NORM) {
        if (R.pos) pos = R.pos[0];       // null where no matrix of the launch is rotated
        if (R.cells) cell = R.cells[0];  // ... or goes to a cache
        if constexpr (STEPS > 1) {
            row.request(R.nx, R.nw, K);
            __builtin_amdgcn_sched_barrier(0);
            request(0, FIRST);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    float rope_c[NP], rope_s[NP];
    bool rotate[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
        rope_c[p] = 1.0f;
        rope_s[p] = 0.0f;
        rotate[p] = false;
    }
    if (lane < NCOLS) {
        const bool rope_epi = m.epi == EPI_ROPE || m.epi == EPI_ROPE_CACHE || m.epi == EPI_ROPE_QCACHE;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int d = (int)((row0 + 2 * p) % R.D);
            rotate[p] = rope_epi && d < R.n_dims;
            if (rotate[p]) rope_coeffs(R, NORM ? pos : R.pos[lane], d >> 1, rope_c[p], rope_s[p]);
        }
        if (!NORM && (m.epi == EPI_ROPE_CACHE || m.epi == EPI_CACHE)) cell = R.cells[lane];
    }
#pragma unroll
    for (int p = 0; p < NP; p++) asm volatile("" : "+v"(rope_c[p]), "+v"(rope_s[p]));
    asm volatile("" : "+v"(cell));

    if constexpr (NORM) {
        if constexpr (STEPS == 1) {
            request(0, FIRST);
            __builtin_amdgcn_sched_barrier(0);
            row.request(R.nx, R.nw, K);
            __builtin_amdgcn_sched_barrier(0);
        }
        row.finish(s_act, K, R.neps, s_norm);
        if constexpr (!G::ORDERED) request(FIRST, STEPS);
        __syncthreads();
        if (!wave_live) return;
        aq = (const int8_t *)s_act;
        ads = (const act_ds *)(s_act + NCOLS * K);
    }

    float acc[RPW][NCOLS];
#pragma unroll
    for (int r = 0; r < RPW; r++)
#pragma unroll
        for (int c = 0; c < NCOLS; c++) acc[r][c] = 0.0f;
    if constexpr (NORM) {
#pragma unroll
        for (int p = 0; p < STEPS; p++) {
            const int c = p * 64 + lane;
            if (p * 64 >= nchunks) break;   // uniform
            if (G::ORDERED && p >= FIRST) request(p, p + 1);
            const typename T::act A = T::load_a(aq, ads, c < nchunks ? c : nchunks - 1);
#pragma unroll
            for (int r = 0; r < RPW; r++) {
                const typename T::chunk now = G::decode(wn[p][r], c);
                const float sum = T::accumulate(acc[r][0], now, A, T::dots(now, A));
                acc[r][0] = c < nchunks ? sum : acc[r][0];
            }
        }
    } else {
        for (int c0 = 0; c0 < nchunks; c0 += 64) {
            const int c = c0 + lane;
            if (c < nchunks) {
                typename T::chunk w[RPW];
#pragma unroll
                for (int r = 0; r < RPW; r++) w[r] = T::load_w(rows[r], L, c);
#pragma unroll
                for (int col = 0; col < NCOLS; col++) {
                    const typename T::act A = T::load_a(aq + (int64_t)col * K, ads + col * nblk, c);
#pragma unroll
                    for (int r = 0; r < RPW; r++) {
                        const chunk_dots d = T::dots(w[r], A);
                        acc[r][col] = T::accumulate(acc[r][col], w[r], A, d);
                    }
                }
            }
        }
    }
    float sv[RPW];
#pragma unroll
    for (int r = 0; r < RPW; r++) sv[r] = 0.0f;
#pragma unroll
    for (int r = 0; r < RPW; r++)
#pragma unroll
        for (int c = 0; c < NCOLS; c++) {
            const float a = wave_sum_dpp(acc[r][c]);
            if (lane == c) sv[r] = a;
        }
    if constexpr (QUANT) {
        __shared__ float s_blk[NCOLS][32];
        if (lane < NCOLS) {
#pragma unroll
            for (int p = 0; p < NP; p++) {
                float y0 = sv[2 * p], y1 = sv[2 * p + 1];
                if (rotate[p]) rope_apply(rope_c[p], rope_s[p], sv[2 * p], sv[2 * p + 1], y0, y1);
                s_blk[lane][wave * RPW + 2 * p] = y0;
                s_blk[lane][wave * RPW + 2 * p + 1] = y1;
            }
        }
        __syncthreads();
        if (wave < NCOLS) {
            const int j = lane & 31;
            const float v = s_blk[wave][j];
            const int64_t g = m.nb1 + (int64_t)R.cells[wave] * (m.N >> 5) + group;
            const kv_place pl = {0, m.nb2};
            int64_t lv, sc;
            if (m.ctype == MI355_Q8_0) {
                kv_block_offsets<MI355_Q8_0>(pl, g, lv, sc);
                kv_store_q8_0_lane32(v, j, (uint8_t *)m.dst, lv, sc, lane < 32);
            } else {
                kv_block_offsets<MI355_Q4_0>(pl, g, lv, sc);
                kv_store_q4_0_lane32(v, j, (uint8_t *)m.dst, lv, sc, lane < 32);
            }
        }
    } else if (lane < NCOLS && row0 + 1 < m.N) {
        const int64_t head = row0 / R.D;
        const int d = (int)(row0 % R.D);
        float y0 = sv[0], y1 = sv[1];
        if (rotate[0]) rope_apply(rope_c[0], rope_s[0], sv[0], sv[1], y0, y1);
        if (m.epi == EPI_ROPE || m.epi == EPI_STORE) {
            float *o = m.dst + lane * m.dst_stride + row0;
            o[0] = y0;
            o[1] = y1;
        } else {
            _Float16 *o = (_Float16 *)((uint8_t *)m.dst + (int64_t)cell * m.nb1 + head * m.nb2) + d;
            o[0] = (_Float16)y0;
            o[1] = (_Float16)y1;
        }
    }
}

// dynamic LDS of the launches below: the group's copy of the activation (LDSA), act_lds_bytes() bytes
extern __shared__ __attribute__((aligned(16))) uint8_t s_act_dyn[];

// bytes of LDS for the group's copy of the activation, or 0 when every wave reads it from memory.  The copy pays when the
// launch has several generations of groups per compute unit (its round trip then hides behind other groups' loads, and the
// activation reads it saves are the larger part of the launch's L2 traffic): output projection 98.9 -> 77.5 us (6.8 TB/s),
// 14336 x 4096 8.6 -> 8.0 us.  One row against one matrix of few rows (wo, ffn_down) has a kernel of its own, gemv_row.hip; the launches of several rows or matrices
// whose groups are all resident at once are one dependent chain per wave, and there the copy's barrier lengthened it (+0.3 to +0.7 us measured).  Up to four activation rows, and
// small enough that eight groups still fit a compute unit.
// Measured and not adopted: splitting K over the four waves of a group (each wave reads a quarter of the activation, partial
// sums meet in LDS at the end) - Q4_K 4096 x 4096 4.9 -> 4.3 us and 14336 x 4096 8.2 -> 7.9 us, but Q6_K slower throughout
// (4096 x 14336 11.2 -> 14.0 us, output projection 80 -> 87 us): its 16-byte pieces per lane then form 256-byte runs.
// Also measured and not adopted: the next step's weights requested before the current step's are used (one step of look-ahead in
// the loop below) - Q4_K 4096 x 14336 10.9 -> 10.7 us, but norm + Q/K/V 10.0 -> 10.8, Q6_K 4096 x 14336 11.9 -> 13.9, wo 4.85 -> 5.1
// and the output projection 70 -> 123 us (decode 557 -> 521 tokens/s).
// Also measured and not adopted: a fixed number of groups (512..1536) that walk the matrix, activation copied to LDS once per
// group, the next block's weights requested before the current one is contracted - bit-identical sums, but 14336 x 4096 Q4_K
// 8.3 -> 9.9..10.9 us and the output projection 50.6 -> 61..77 us: many short-lived waves keep more loads in flight than few
// long-lived ones with one block of look-ahead.
inline size_t act_lds_bytes(int ncols, int64_t K, int64_t groups) {
    const int64_t bytes = (int64_t)ncols * (K + K / 4);
    return (groups >= 1536 && ncols <= 4 && bytes <= 20480) ? (size_t)bytes : 0;
}

inline int check_gemv_args(const char *who, int type, const void *W, int64_t N, int64_t K, int64_t dst_stride) {
    MI355_REQUIRE(is_weight_type(type), "%s: unsupported weight type %d", who, type);
    MI355_REQUIRE(N > 0 && K > 0 && K < (int64_t(1) << 30), "%s: bad shape N=%lld K=%lld", who, (long long)N, (long long)K);
    MI355_REQUIRE(K % type_block_elems(type) == 0, "%s: K=%lld is not a multiple of the block size", who, (long long)K);
    MI355_REQUIRE(dst_stride >= N, "%s: dst_stride < N", who);
    MI355_REQUIRE(layout_aligned(W, make_row_layout(type, K)), "%s: weight rows are not 16-byte aligned (K=%lld)", who, (long long)K);
    return MI355_OK;
}

}  // namespace mi355
