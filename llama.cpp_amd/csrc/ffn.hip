// The feed-forward half of a decoded token (llm_build_ffn with LLM_FFN_SILU / LLM_FFN_PAR, src/llama.cpp:280-320):
//   k_gemv_gate_up_blk   ffn_gate, ffn_up, SiLU(gate) * up and the Q8_1 quantization of the product in one launch with no step
//                        between groups: a group owns the 32 output rows of one Q8_1 block in BOTH matrices.
// Measured and not adopted: the same launch continued, past a grid-wide step (per-group flags polled with device-scope loads, the
// wait bounded by the wall clock), with ffn_down + residual, every wave requesting its ffn_down rows before it waits - bit-identical
// to the two launches, but 33.1 / 34.9 us (Q4_K / Q6_K ffn_down) against 15.3 + 10.6 / 11.5 us on the 8B shape: a compute unit's
// vector memory requests complete in order, so the flag polls queue behind the unit's own weight requests and the step costs as
// much as the stream it was meant to hide.
// Row sums are formed exactly as in gemv_body (gemv.hip): same lane-to-chunk mapping, same step order, same wave reduction, so
// every result holds the bits of the separate launches (ggml_compute_forward_mul_mat, ggml-cpu.c:7443-7635, with
// ggml_vec_dot_q*_q8_*; UNARY(SILU) and MUL :6646-6683, 5142-5211; quantize_row_q8_1_ref, ggml-quants.c:220-253).
#include "common.hpp"
#include "qdot.hpp"
#include "norm_quant.hpp"
#include "ffn.hpp"

namespace mi355 {

extern __shared__ __attribute__((aligned(16))) uint8_t s_ffn_dyn[];

// Eight waves per group; rows of each matrix a wave has in flight.  The types with the largest chunks walk their four rows in two or four rounds, or their registers would not leave room
// for two groups per compute unit: 14336 x 4096, us, one token, Q4_K four rows 17.3 (spilled), two 12.9; Q6_K two or three tokens two rows 23.1 / 27.1, one 20.6 / 24.0, but one and four
// tokens 19.2 / 29.9 and 19.0 / 31.6 (28672 x 8192: 94.6 and 105.3).
constexpr int GU_WAVES = 8;
constexpr int gu_rows_in_flight(int type, int ncols) {
    return type == MI355_Q5_K || (type == MI355_Q6_K && (ncols == 2 || ncols == 3)) ? 1 : type == MI355_Q4_K || type == MI355_Q6_K ? 2 : 4;
}
// Rows are used in the order their loads return, and a register goes to its row's next step or round as soon as it is used.  Not for one token of the other types, whose step is
// some twenty instructions: requesting a step's rows together when the one before is done is as fast or faster there (28672 x 8192, us: Q4_0 41.4 against 42.4, Q8_0 84.9 against
// 88.1, IQ4_XS 48.5 against 54.4).
constexpr bool gu_ahead(int type, int ncols) { return ncols > 1 || type == MI355_Q4_K || type == MI355_Q5_K || type == MI355_Q6_K; }

// Wave w of the group: rows 32 b + RPM w .. + RPM - 1 of gate and of up (RPM = 32 / WAVES), R rows of each in flight; the
// block's 32 values of every activation row meet in s_g / s_u and are quantized by the group's first lanes.  The activation is
// requested first and the first round's weights behind it, before it goes to LDS.  COH: the quantized block is stored with device scope.
// The 66 MB of an 8B layer's two matrices take 12.2 us as one matrix with a wave per row (k_gemv_row); with all of a wave's eight rows requested at once and used in the order the
// compiler chose - the scales of every row decoded first, 400 of 600 instructions behind the last row's arrival, a store per row - this launch took 14.4, now 12.9
// (a token 1508 -> 1472).  Three tokens 62.7 -> 20.8 (spilled registers), Q5_K 20.3 -> 17.6, Q6_K 20.2 -> 18.9, Q4_0 with three tokens 20.8 -> 16.5.
template <int TYPE, int NCOLS, int WAVES, int R, bool COH>
__device__ __forceinline__ void gate_up_blk_phase(const uint8_t *__restrict__ Wg, const uint8_t *__restrict__ Wu, const int8_t *__restrict__ aq,
                                                  const act_ds *__restrict__ ads, int K, float *__restrict__ gate, float *__restrict__ up,
                                                  int64_t out_stride, int8_t *__restrict__ act_q, act_ds *__restrict__ act_s, int n,
                                                  uint8_t *s_act, float (*s_g)[32], float (*s_u)[32]) {
    typedef wq<TYPE> T;
    constexpr int RPM = 32 / WAVES;            // rows of each matrix per wave
    static_assert(RPM % R == 0, "rows per wave are walked in rounds of R");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t blk = blockIdx.x;
    const row_layout L = make_row_layout(TYPE, K);
    const int nchunks = K / T::CHUNK;
    const int nblk = K >> 5;
    const int64_t row0 = blk * 32 + wave * RPM;
    typedef late_chunk<TYPE> G;
    constexpr bool AHEAD = gu_ahead(TYPE, NCOLS);
    // the first round's weights of step 0 are requested behind the activation
    const uint8_t *rows[2 * R];
    typename G::raw w[2 * R];
    auto row_of = [&](int round, int r) { return (r < R ? Wg : Wu) + (row0 + round * R + (r < R ? r : r - R)) * L.row_bytes; };
#pragma unroll
    for (int r = 0; r < 2 * R; r++) rows[r] = row_of(0, r);
    const int c_first = lane < nchunks ? lane : nchunks - 1;
    int8_t *s_q = (int8_t *)s_act;
    act_ds *s_ds = (act_ds *)(s_act + NCOLS * K);
    act_copy<NCOLS, 64 * WAVES> copy;
    copy.request(aq, ads, K);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 2 * R; r++) {
        w[r] = G::load(rows[r], L, c_first);
        if constexpr (AHEAD && G::ORDERED) __builtin_amdgcn_sched_barrier(0);   // a row must not wait for pieces of a later one
    }
    copy.commit(s_act, aq, ads, K);
    __syncthreads();
    float acc[2 * R][NCOLS];
    // one step of every row.  next(r): requests what the row's register holds next
    auto step = [&](int c, bool live, auto next) {
        if constexpr (NCOLS == 1 && AHEAD) {
            const typename T::act A = T::load_a(s_q, s_ds, c);
#pragma unroll
            for (int r = 0; r < 2 * R; r++) {
                const typename T::chunk now = G::decode(w[r], c);
                const float sum = T::accumulate(acc[r][0], now, A, T::dots(now, A));
                acc[r][0] = live ? sum : acc[r][0];
                next(r);
                __builtin_amdgcn_sched_barrier(0);   // (left to itself the compiler decodes the scales of all rows first, and most of the step's instructions wait for the last row)
            }
        } else {
            typename T::chunk now[2 * R];
#pragma unroll
            for (int r = 0; r < 2 * R; r++) {
                now[r] = G::decode(w[r], c);
                next(r);
            }
#pragma unroll
            for (int col = 0; col < NCOLS; col++) {
                const typename T::act A = T::load_a(s_q + (int64_t)col * K, s_ds + col * nblk, c);
#pragma unroll
                for (int r = 0; r < 2 * R; r++) {
                    const float sum = T::accumulate(acc[r][col], now[r], A, T::dots(now[r], A));
                    acc[r][col] = live ? sum : acc[r][col];
                }
            }
        }
    };
#pragma unroll
    for (int round = 0; round < RPM / R; round++) {
#pragma unroll
        for (int r = 0; r < 2 * R; r++)
#pragma unroll
            for (int c = 0; c < NCOLS; c++) acc[r][c] = 0.0f;
        if constexpr (AHEAD) {
            int c0 = 0;
            for (; c0 + 64 < nchunks; c0 += 64) {
                const int after = c0 + 64 + lane < nchunks ? c0 + 64 + lane : nchunks - 1;
                step(c0 + lane, true, [&](int r) { w[r] = G::load(rows[r], L, after); });
            }
            const int c = c0 + lane;
            step(c < nchunks ? c : nchunks - 1, c < nchunks, [&](int r) {
                if (round + 1 < RPM / R) {
                    rows[r] = row_of(round + 1, r);
                    w[r] = G::load(rows[r], L, c_first);
                }
            });
        } else {
#pragma unroll
            for (int r = 0; r < 2 * R; r++) rows[r] = row_of(round, r);
            for (int c0 = 0; c0 < nchunks; c0 += 64) {
                const int c = c0 + lane;
                if (c < nchunks) {
                    if (round > 0 || c0 > 0) {
#pragma unroll
                        for (int r = 0; r < 2 * R; r++) w[r] = G::load(rows[r], L, c);
                    }
                    step(c, true, [](int) {});
                }
            }
        }
        // lane r keeps row r's sum and stores it
#pragma unroll
        for (int col = 0; col < NCOLS; col++) {
            float mine = 0.0f;
#pragma unroll
            for (int r = 0; r < 2 * R; r++) {
                const float sum = wave_sum_dpp(acc[r][col]);
                mine = lane == r ? sum : mine;
            }
            const int j = wave * RPM + round * R + (lane < R ? lane : lane - R);   // row inside the block
            if (lane < R) { s_g[col][j] = mine; gate[col * out_stride + blk * 32 + j] = mine; }
            else if (lane < 2 * R) { s_u[col][j] = mine; up[col * out_stride + blk * 32 + j] = mine; }
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < 32 * NCOLS; idx += 64 * WAVES) {   // whole aligned groups of 32 lanes
        const int col = idx >> 5, j = idx & 31;
        const float h = silu_fast(s_g[col][j]) * s_u[col][j];
        quantize_lane32<COH>(h, act_q + (int64_t)col * n, act_s + (int64_t)col * (n >> 5), blk * 32 + j);
    }
}

template <int TYPE, int NCOLS, int WAVES, int R>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(NCOLS == 1 ? 4 : 1, 8)))
k_gemv_gate_up_blk(const uint8_t *__restrict__ Wg, const uint8_t *__restrict__ Wu, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int K,
                   float *__restrict__ gate, float *__restrict__ up, int64_t out_stride, int8_t *__restrict__ act_q, act_ds *__restrict__ act_s, int n) {
    __shared__ float s_g[NCOLS][32], s_u[NCOLS][32];
    gate_up_blk_phase<TYPE, NCOLS, WAVES, R, false>(Wg, Wu, aq, ads, K, gate, up, out_stride, act_q, act_s, n, s_ffn_dyn, s_g, s_u);
}

int launch_gate_up_blk(hipStream_t s, int type, const void *w_gate, const void *w_up, const int8_t *aq, const act_ds *ads, int64_t K, int64_t B,
                       float *gate, float *up, int64_t out_stride, void *act_out, int64_t N) {
    const size_t lds = (size_t)(B * (K + K / 4));
    int8_t *oq = (int8_t *)act_out;
    act_ds *os = (act_ds *)(oq + B * N);
    const dim3 grid((unsigned)(N / 32));
#define MI355_BLK_ARGS grid, dim3(64 * GU_WAVES), lds, s, (const uint8_t *)w_gate, (const uint8_t *)w_up, aq, ads, (int)K, gate, up, out_stride, oq, os, (int)N
#define MI355_BLK_LAUNCH(TY)                                                                                        \
    switch (B) {                                                                                                    \
        case 1: MI355_LAUNCH((k_gemv_gate_up_blk<TY, 1, GU_WAVES, gu_rows_in_flight(TY, 1)>), MI355_BLK_ARGS); break;  \
        case 2: MI355_LAUNCH((k_gemv_gate_up_blk<TY, 2, GU_WAVES, gu_rows_in_flight(TY, 2)>), MI355_BLK_ARGS); break;  \
        case 3: MI355_LAUNCH((k_gemv_gate_up_blk<TY, 3, GU_WAVES, gu_rows_in_flight(TY, 3)>), MI355_BLK_ARGS); break;  \
        default: MI355_LAUNCH((k_gemv_gate_up_blk<TY, 4, GU_WAVES, gu_rows_in_flight(TY, 4)>), MI355_BLK_ARGS); break; \
    }
    MI355_WEIGHT_TYPE_SWITCH(type, MI355_BLK_LAUNCH)
#undef MI355_BLK_LAUNCH
#undef MI355_BLK_ARGS
    return launch_status("k_gemv_gate_up_blk");
}

// The same launch for the experts of a mixture-of-experts layer (llm_build_moe_ffn, src/llama.cpp:417-538: MUL_MAT_ID(up),
// MUL_MAT_ID(gate), SILU, MUL): blockIdx.y = slot = t * n_used + e, the expert read on the device as k_gemv_id does, one activation
// row per slot.  gate / up: f32 [slots][N]; the quantized product: rows of N per slot.
template <int TYPE, int WAVES, int R>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_gemv_gate_up_blk_id(const uint8_t *__restrict__ as_gate, const uint8_t *__restrict__ as_up, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads,
                      const int32_t *__restrict__ ids, int64_t ids_stride, int K, float *__restrict__ gate, float *__restrict__ up,
                      int8_t *__restrict__ act_q, act_ds *__restrict__ act_s, int n, int64_t n_expert, int64_t n_used, int64_t nb1) {
    __shared__ float s_g[1][32], s_u[1][32];
    const int64_t slot = blockIdx.y, t = slot / n_used, e = slot % n_used;
    int64_t ex = ids[t * ids_stride + e];
    ex = ex < 0 ? 0 : (ex >= n_expert ? n_expert - 1 : ex);   // never index outside the expert stack
    const int64_t arow = t * nb1 + e % nb1;
    const row_layout L = make_row_layout(TYPE, K);
    const int64_t expert_bytes = (int64_t)n * L.row_bytes;
    gate_up_blk_phase<TYPE, 1, WAVES, R, false>(as_gate + ex * expert_bytes, as_up + ex * expert_bytes, aq + arow * K, ads + arow * (K >> 5), K,
                                                gate + slot * n, up + slot * n, n, act_q + slot * n, act_s + slot * (n >> 5), n, s_ffn_dyn, s_g, s_u);
}

int launch_gate_up_blk_id(hipStream_t s, int type, const void *as_gate, const void *as_up, const int8_t *aq, const act_ds *ads, const int32_t *ids,
                          int64_t ids_stride, int64_t K, float *gate, float *up, void *act_out, int64_t N, int64_t n_expert, int64_t n_used, int64_t nb1,
                          int64_t T) {
    const size_t lds = (size_t)(K + K / 4);
    const int64_t slots = n_used * T;
    int8_t *oq = (int8_t *)act_out;
    act_ds *os = (act_ds *)(oq + slots * N);
    const dim3 grid((unsigned)(N / 32), (unsigned)slots);
#define MI355_BLK_ID_LAUNCH(TY)                                                                                                                          \
    MI355_LAUNCH((k_gemv_gate_up_blk_id<TY, GU_WAVES, gu_rows_in_flight(TY, 1)>), grid, dim3(64 * GU_WAVES), lds, s, (const uint8_t *)as_gate,              \
                 (const uint8_t *)as_up, aq, ads, ids, ids_stride, (int)K, gate, up, oq, os, (int)N, n_expert, n_used, nb1);
    MI355_WEIGHT_TYPE_SWITCH(type, MI355_BLK_ID_LAUNCH)
#undef MI355_BLK_ID_LAUNCH
    return launch_status("k_gemv_gate_up_blk_id");
}

}  // namespace mi355
