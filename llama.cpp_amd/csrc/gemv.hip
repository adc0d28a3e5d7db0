// Bandwidth-bound quantized GEMV (batch 1..8): dst[b][n] = sum_k W[n][k] * x[b][k] (+ residual).
//
// One wave owns RPW consecutive weight rows and walks them in steps of 64 chunks: every lane
// issues 16-byte streaming loads to consecutive addresses across the wave, so HBM sees long
// linear bursts.  The activation chunk (already Q8_1-quantized, L2 resident) is loaded once
// per step and reused for all RPW rows and all NCOLS activation rows.  Integer dots use
// v_dot4_i32_i8; scales are applied in f32; the wave reduces with cross-lane shuffles.
//
// One launch can serve up to four weight matrices that share the activation (Q/K/V, gate/up):
// the groups of all matrices are laid end to end in the grid, which turns three short launches
// into one long enough to fill the chip.  An optional residual is added in the epilogue.
#include "ffn.hpp"
#include "gemv_body.hpp"
#include "gemv_row.hpp"

#include <math.h>
#include <stdlib.h>

namespace mi355 {

template <int NCOLS, int RPW, bool COH = false, bool LDSA = false>
__device__ __forceinline__ void gemv_dispatch(const gemv_item &m, int group, const int8_t *__restrict__ aq,
                                              const act_ds *__restrict__ ads, int K) {
#define MI355_BODY(TY) gemv_body<TY, NCOLS, RPW, false, COH, LDSA>(m, group, aq, ads, K, nullptr, s_act_dyn);
    MI355_WEIGHT_TYPE_SWITCH(m.type, MI355_BODY)   // uniform over the group
#undef MI355_BODY
}

// single matrix, type known at compile time (smallest code, used by mi355_mul_mat_vec_q)
template <int TYPE, int NCOLS, int RPW, bool LDSA>
__global__ void __launch_bounds__(256) k_gemv_q(gemv_item m, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int K) {
    gemv_body<TYPE, NCOLS, RPW, false, false, LDSA>(m, blockIdx.x, aq, ads, K, nullptr, s_act_dyn);
}

// several matrices sharing one activation
template <int NCOLS, int RPW, bool LDSA>
__global__ void __launch_bounds__(256) k_gemv_multi(gemv_batch b, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int K) {
    const int g = blockIdx.x;
    int i = 0;
#pragma unroll
    for (int j = 1; j < 4; j++)
        if (j < b.n && g >= b.it[j].first_group) i = j;
    gemv_dispatch<NCOLS, RPW, false, LDSA>(b.it[i], g - b.it[i].first_group, aq, ads, K);
}

// ---- a launch whose last-arriving groups also do the nodes that follow the product ------------
// Every group stores its rows with device scope and waits for those stores (an explicit vmcnt wait), then
// one thread takes a ticket from the counter of its 32-row block.  The group that draws the last
// ticket of a block knows that all of the block's rows have been written, reads them back with
// device-scope loads, finishes the follow-up nodes and re-arms the counter for the next launch.  No
// cache-wide fence is involved (a device-scope fence per group writes back and invalidates the
// whole L2 and made a decoded token 10x slower), counters are shared by 8 groups only (one counter
// for a whole launch serialises ~1000 device-scope atomics), and nobody waits for anybody, so
// there is nothing that could hang.
// The same scheme for the RMS norm that follows wo / ffn_down (last group of the whole launch normalises the row; tickets on
// two levels) was measured and dropped: store acknowledgement, two dependent device-scope atomics and the device-scope
// read-back are ~2 us each and all on the critical path of a 4-10 us launch, 12 us in total against 5.8 us for the separate
// norm launch.  Here the block tails overlap with the other blocks' products and only the last one is exposed.
struct gemv_tail {
    unsigned *counters;     // one per 32-row block; zero before the first launch, left zero by every launch
    int8_t *act_q;          // quantized output, split activation layout
    act_ds *act_s;
    const float *x2;        // rows of the second matrix (up), same stride as the first
    int n;                  // elements per output row (N of the matrices)
};

__device__ __forceinline__ float load_coherent(const float *p) {   // bypasses caches that other XCDs cannot invalidate
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// gate and up projections (llm_build_ffn, src/llama.cpp:280-320) with UNARY(SILU), MUL and the Q8_1 quantization of
// the product done per 32-row block by whichever of the block's 8 groups (4 per matrix, 8 rows each) finishes last
template <int NCOLS, bool LDSA>
__global__ void __launch_bounds__(256) k_gemv_gate_up(gemv_batch b, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int K, gemv_tail t) {
    __shared__ unsigned s_ticket;
    const int g = blockIdx.x;
    const int i = g >= b.it[1].first_group ? 1 : 0;
    const int group = g - b.it[i].first_group;
    gemv_dispatch<NCOLS, 2, true, LDSA>(b.it[i], group, aq, ads, K);
    // Every wave waits until its device-scope stores have been acknowledged before it reaches the barrier: the
    // barrier's own wait covers LDS and scalar loads only, and a ticket that overtakes a row store would let the
    // last group read that row too early.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const int block = group >> 2;   // 8 rows per group, 32 rows per quantization block
    if (threadIdx.x == 0) s_ticket = atomicAdd(t.counters + block, 1u);
    __syncthreads();
    if (s_ticket != 7u) return;   // uniform over the group
    if (threadIdx.x == 0) t.counters[block] = 0;
    const int tid = threadIdx.x;
    for (int idx = tid; idx < 32 * NCOLS; idx += 256) {   // NCOLS <= 4: whole waves, aligned groups of 32 lanes
        const int col = idx >> 5, j = idx & 31;
        const int64_t row = (int64_t)block * 32 + j;
        const float gv = load_coherent(b.it[0].dst + col * b.it[0].dst_stride + row);
        const float uv = load_coherent(t.x2 + col * b.it[0].dst_stride + row);
        const float h = silu_fast(gv) * uv;
        quantize_lane32<false>(h, t.act_q + (int64_t)col * t.n, t.act_s + (int64_t)col * (t.n >> 5), row);
    }
}

// MUL_MAT_ID, one activation row per expert slot: blockIdx.y = slot = t * n_used + e.  The
// expert id is read on the device, so no host synchronisation is needed to route tokens.
template <int TYPE, int RPW, bool LDSA>
__global__ void __launch_bounds__(256) k_gemv_id(const uint8_t *__restrict__ as, const int8_t *__restrict__ aq,
                                                 const act_ds *__restrict__ ads, const int32_t *__restrict__ ids,
                                                 int64_t ids_stride, float *__restrict__ dst, int64_t N, int K,
                                                 int64_t n_expert, int64_t n_used, int64_t nb1) {
    const int64_t slot = blockIdx.y, t = slot / n_used, e = slot % n_used;
    int64_t ex = ids[t * ids_stride + e];
    ex = ex < 0 ? 0 : (ex >= n_expert ? n_expert - 1 : ex);   // never index outside the expert stack
    const int64_t arow = t * nb1 + e % nb1;
    const row_layout L = make_row_layout(TYPE, K);
    gemv_item m;
    m.W = as + ex * N * L.row_bytes;
    m.dst = dst + slot * N;
    m.residual = nullptr;
    m.N = N;
    m.dst_stride = N;
    m.type = TYPE;
    m.first_group = 0;
    gemv_body<TYPE, 1, RPW, false, false, LDSA>(m, blockIdx.x, aq + arow * K, ads + arow * (K >> 5), K, nullptr, s_act_dyn);
}

// Same routing for expert stacks at an odd address (byte loads): one wave per (row, slot).
template <int TYPE>
__global__ void __launch_bounds__(64) k_gemv_id_unaligned(const uint8_t *__restrict__ as, const int8_t *__restrict__ aq,
                                                          const act_ds *__restrict__ ads, const int32_t *__restrict__ ids,
                                                          int64_t ids_stride, float *__restrict__ dst, int64_t N, int64_t K,
                                                          int64_t n_expert, int64_t n_used, int64_t nb1, row_layout L) {
    const int64_t row = blockIdx.x, slot = blockIdx.y, t = slot / n_used, e = slot % n_used;
    int64_t ex = ids[t * ids_stride + e];
    ex = ex < 0 ? 0 : (ex >= n_expert ? n_expert - 1 : ex);
    const int64_t arow = t * nb1 + e % nb1;
    const uint8_t *wrow = as + (ex * N + row) * L.row_bytes;
    const int8_t *q = aq + arow * K;
    const act_ds *ds = ads + arow * (K >> 5);
    float acc = 0.0f;
    for (int64_t i = threadIdx.x; i < K; i += 64) acc += weight_value<TYPE>(wrow, L, i) * (ds[i >> 5].d * (float)q[i]);
    acc = wave_sum(acc);
    if (threadIdx.x == 0) dst[slot * N + row] = acc;
}

// Parity dump of the integer granule dots (one wave per row, activation row 0).
template <int TYPE>
__global__ void __launch_bounds__(64) k_block_dots(const uint8_t *__restrict__ W, const int8_t *__restrict__ aq,
                                                   const act_ds *__restrict__ ads, int32_t *__restrict__ out, int64_t N, int K) {
    typedef wq<TYPE> T;
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const row_layout L = make_row_layout(TYPE, K);
    const int nchunks = K / T::CHUNK;
    const int ngran = TYPE == MI355_Q6_K ? K / 16 : K / 32;
    const uint8_t *wrow = W + row * L.row_bytes;
    for (int c0 = 0; c0 < nchunks; c0 += 64) {
        const int c = c0 + lane;
        const bool live = c < nchunks;
        const int cc = live ? c : 0;
        const typename T::chunk w = T::load_w(wrow, L, cc);
        const typename T::act A = T::load_a(aq, ads, cc);
        const chunk_dots d = T::dots(w, A);
        if (!live) continue;
        if constexpr (T::CHUNK == 32 && TYPE != MI355_Q6_K) {   // one 32-element block per chunk
            out[row * ngran + c] = d.i0;
        } else if constexpr (TYPE == MI355_Q4_K || TYPE == MI355_Q5_K) {   // chunk c = sub-blocks 2c and 2c+1 of the row
            out[row * ngran + 2 * c] = d.i0;
            out[row * ngran + 2 * c + 1] = d.i1;
        } else {   // Q6_K: 16 granules per super-block
            const int sb = c >> 3, ccc = c & 7, hf = ccc >> 2, r = ccc & 3;
            const int gi = 8 * hf + 2 * (r >> 1) + (r & 1);
            out[row * ngran + sb * 16 + gi] = d.i0;
            out[row * ngran + sb * 16 + gi + 4] = d.i1;
        }
    }
}

// rows per wave: enough waves to cover every SIMD a few times over, then amortise the
// activation reads over more rows.
static int pick_rpw(int64_t total_rows) {
    if (total_rows >= 32768) return 4;
    if (total_rows >= 8192) return 2;
    return 1;
}

template <int NCOLS>
static void launch_multi(int rpw, hipStream_t s, const gemv_batch &b, unsigned grid, const int8_t *aq, const act_ds *ads, int K) {
    if constexpr (NCOLS <= 4) {
        if (const size_t lds = act_lds_bytes(NCOLS, K, grid)) {
            if (rpw == 1) MI355_LAUNCH((k_gemv_multi<NCOLS, 1, true>), dim3(grid), dim3(256), lds, s, b, aq, ads, K);
            else if (rpw == 2) MI355_LAUNCH((k_gemv_multi<NCOLS, 2, true>), dim3(grid), dim3(256), lds, s, b, aq, ads, K);
            else MI355_LAUNCH((k_gemv_multi<NCOLS, 4, true>), dim3(grid), dim3(256), lds, s, b, aq, ads, K);
            return;
        }
    }
    if (rpw == 1) MI355_LAUNCH((k_gemv_multi<NCOLS, 1, false>), dim3(grid), dim3(256), 0, s, b, aq, ads, K);
    else if (rpw == 2) MI355_LAUNCH((k_gemv_multi<NCOLS, 2, false>), dim3(grid), dim3(256), 0, s, b, aq, ads, K);
    else MI355_LAUNCH((k_gemv_multi<NCOLS, 4, false>), dim3(grid), dim3(256), 0, s, b, aq, ads, K);
}

template <int TYPE, int NCOLS>
static void launch_single(int rpw, hipStream_t s, const gemv_item &m, unsigned grid, const int8_t *aq, const act_ds *ads, int K) {
    if constexpr (NCOLS <= 4) {
        if (const size_t lds = act_lds_bytes(NCOLS, K, grid)) {
            if (rpw == 1) MI355_LAUNCH((k_gemv_q<TYPE, NCOLS, 1, true>), dim3(grid), dim3(256), lds, s, m, aq, ads, K);
            else if (rpw == 2) MI355_LAUNCH((k_gemv_q<TYPE, NCOLS, 2, true>), dim3(grid), dim3(256), lds, s, m, aq, ads, K);
            else MI355_LAUNCH((k_gemv_q<TYPE, NCOLS, 4, true>), dim3(grid), dim3(256), lds, s, m, aq, ads, K);
            return;
        }
    }
    if (rpw == 1) MI355_LAUNCH((k_gemv_q<TYPE, NCOLS, 1, false>), dim3(grid), dim3(256), 0, s, m, aq, ads, K);
    else if (rpw == 2) MI355_LAUNCH((k_gemv_q<TYPE, NCOLS, 2, false>), dim3(grid), dim3(256), 0, s, m, aq, ads, K);
    else MI355_LAUNCH((k_gemv_q<TYPE, NCOLS, 4, false>), dim3(grid), dim3(256), 0, s, m, aq, ads, K);
}

template <int TYPE>
static void launch_single_cols(int rpw, int64_t B, hipStream_t s, const gemv_item &m, unsigned grid, const int8_t *aq, const act_ds *ads, int K) {
    switch (B) {
        case 1: launch_single<TYPE, 1>(rpw, s, m, grid, aq, ads, K); break;
        case 2: launch_single<TYPE, 2>(rpw, s, m, grid, aq, ads, K); break;
        case 3: launch_single<TYPE, 3>(rpw, s, m, grid, aq, ads, K); break;
        case 4: launch_single<TYPE, 4>(rpw, s, m, grid, aq, ads, K); break;
        case 5: launch_single<TYPE, 5>(rpw, s, m, grid, aq, ads, K); break;
        case 6: launch_single<TYPE, 6>(rpw, s, m, grid, aq, ads, K); break;
        case 7: launch_single<TYPE, 7>(rpw, s, m, grid, aq, ads, K); break;
        default: launch_single<TYPE, 8>(rpw, s, m, grid, aq, ads, K); break;
    }
}

}  // namespace mi355

using namespace mi355;

extern "C" {

int mi355_mul_mat_vec_q(void *stream, int type, const void *W, const void *act, float *dst, int64_t N, int64_t K,
                        int64_t B, int64_t dst_stride) {
    mi355_gemv_mat m = {type, W, N, dst, dst_stride, nullptr};
    return mi355_mul_mat_vec_q_multi(stream, 1, &m, act, K, B);
}

int mi355_mul_mat_vec_q_multi(void *stream, int n_mats, const mi355_gemv_mat *mats, const void *act, int64_t K, int64_t B) {
    MI355_REQUIRE(n_mats >= 1 && n_mats <= 4, "mul_mat_vec_q_multi: 1..4 matrices per launch, got %d", n_mats);
    MI355_REQUIRE(B >= 1 && B <= 32, "mul_mat_vec_q: batch %lld outside 1..32", (long long)B);
    MI355_REQUIRE(((uintptr_t)act & 15) == 0, "mul_mat_vec_q: activation workspace is not 16-byte aligned");
    int64_t total_rows = 0;
    bool loadable = true;
    for (int i = 0; i < n_mats; i++) {
        MI355_REQUIRE(is_weight_type(mats[i].type) && K > 0 && K % type_block_elems(mats[i].type) == 0, "mul_mat_vec_q: unsupported type %d or K=%lld not a multiple of its block size", mats[i].type, (long long)K);
        MI355_REQUIRE(mats[i].N > 0 && mats[i].dst_stride >= mats[i].N, "mul_mat_vec_q: bad shape");
        MI355_REQUIRE(K < (int64_t(1) << 30) || !layout_aligned(mats[i].W, make_row_layout(mats[i].type, K)), "mul_mat_vec_q: bad shape K=%lld", (long long)K);
        loadable = loadable && layout_loadable(mats[i].W) && K < (int64_t(1) << 30);
        total_rows += mats[i].N;
    }
    if (!loadable) {   // a matrix at an odd address, rows of 2^30 elements and more: byte-load kernel, one matrix at a time
        for (int i = 0; i < n_mats; i++) {
            int rc = gemv_unaligned((hipStream_t)stream, mats[i].type, mats[i].W, act, mats[i].dst, mats[i].residual, mats[i].N, K, B, mats[i].dst_stride);
            if (rc != MI355_OK) return rc;
        }
        return MI355_OK;
    }
    // From five activation rows on the matrix-core kernel (skinny.hip) is ahead wherever it supports the product; a single
    // Q4_0/Q8_0/Q4_K matrix already at four (14336 x 4096 Q4_K: 14.3 -> 12.0 us, 4096 x 14336: 18.0 -> 14.6 us).
    if (B >= 5 || (B == 4 && n_mats == 1 && mats[0].type != MI355_Q6_K)) {
        bool ok = true;
        for (int i = 0; i < n_mats; i++) ok = ok && mi355_mul_mat_skinny_supported(mats[i].type, mats[i].W, K, B);
        if (ok) {
            for (int i = 0; i < n_mats; i++) {
                int rc = mi355_mul_mat_skinny(stream, mats[i].type, mats[i].W, act, mats[i].dst, mats[i].residual, mats[i].N, K, B, mats[i].dst_stride, nullptr, 0);
                if (rc != MI355_OK) return rc;
            }
            return MI355_OK;
        }
    }
    MI355_REQUIRE(B <= 8, "mul_mat_vec_q: batch %lld needs the matrix-core kernel, which does not support this product", (long long)B);
    int rpw = pick_rpw(total_rows);
    if (B > 4 && rpw > 2) rpw = 2;   // keep the accumulator tile in registers
    {   // per-type corrections, measured on the 8B shapes
        bool any_q6 = false, all_q4k = true;
        for (int i = 0; i < n_mats; i++) {
            any_q6 = any_q6 || mats[i].type == MI355_Q6_K;
            all_q4k = all_q4k && mats[i].type == MI355_Q4_K;
        }
        if (any_q6 && rpw > 2) rpw = 2;                   // 128256 x 4096 Q6_K: 79.5 -> 69.3 us with two rows per wave
        if (all_q4k && rpw == 1 && K >= 8192) rpw = 2;    // 4096 x 14336 Q4_K: 11.4 -> 10.6 us (half the activation reads)
    }
    gemv_batch b;
    b.n = n_mats;
    int64_t groups = 0;
    for (int i = 0; i < 4; i++) {
        const mi355_gemv_mat &src = mats[i < n_mats ? i : 0];
        b.it[i].W = (const uint8_t *)src.W;
        b.it[i].dst = src.dst;
        b.it[i].residual = src.residual;
        b.it[i].N = src.N;
        b.it[i].dst_stride = src.dst_stride;
        b.it[i].type = src.type;
        b.it[i].first_group = (int)groups;
        b.it[i].epi = EPI_STORE;
        b.it[i].nb1 = b.it[i].nb2 = 0;
        if (i < n_mats) groups += (src.N + 4 * rpw - 1) / (4 * rpw);
    }
    MI355_REQUIRE(groups < 0x7fffffff, "mul_mat_vec_q: too many rows for one launch");
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + B * K);
    if (n_mats == 1 && B == 1 && gemv_row_serves(mats[0].N, K))
        return launch_gemv_row(s, mats[0].type, mats[0].W, aq, ads, mats[0].dst, mats[0].residual, mats[0].N, K);
    if (n_mats == 1) {
#define MI355_SINGLE_LAUNCH(TY) launch_single_cols<TY>(rpw, B, s, b.it[0], (unsigned)groups, aq, ads, (int)K);
        MI355_WEIGHT_TYPE_SWITCH(mats[0].type, MI355_SINGLE_LAUNCH)
#undef MI355_SINGLE_LAUNCH
        return launch_status("k_gemv_q");
    }
    switch (B) {
        case 1: launch_multi<1>(rpw, s, b, (unsigned)groups, aq, ads, (int)K); break;
        case 2: launch_multi<2>(rpw, s, b, (unsigned)groups, aq, ads, (int)K); break;
        case 3: launch_multi<3>(rpw, s, b, (unsigned)groups, aq, ads, (int)K); break;
        case 4: launch_multi<4>(rpw, s, b, (unsigned)groups, aq, ads, (int)K); break;
        default:
            // wider batches: one launch per matrix (register budget of the type switch)
            for (int i = 0; i < n_mats; i++) {
                mi355_gemv_mat one = mats[i];
                int rc = mi355_mul_mat_vec_q_multi(stream, 1, &one, act, K, B);
                if (rc != MI355_OK) return rc;
            }
            return MI355_OK;
    }
    return launch_status("k_gemv_multi");
}

int mi355_ffn_gate_up_swiglu(void *stream, int type_gate, const void *w_gate, int type_up, const void *w_up, const void *act, float *gate,
                             float *up, int64_t out_stride, void *act_out, unsigned *counters, int64_t N, int64_t K, int64_t B) {
    MI355_REQUIRE(B >= 1 && B <= 4, "ffn_gate_up_swiglu: batch %lld outside 1..4", (long long)B);
    MI355_REQUIRE(N > 0 && N % 32 == 0 && out_stride >= N, "ffn_gate_up_swiglu: N=%lld must be a positive multiple of 32 and fit the row stride", (long long)N);
    MI355_REQUIRE(((uintptr_t)act & 15) == 0 && ((uintptr_t)act_out & 15) == 0 && counters != nullptr, "ffn_gate_up_swiglu: misaligned or missing operands");
    int rc = check_gemv_args("ffn_gate_up_swiglu", type_gate, w_gate, N, K, out_stride);
    if (rc != MI355_OK) return rc;
    rc = check_gemv_args("ffn_gate_up_swiglu", type_up, w_up, N, K, out_stride);
    if (rc != MI355_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + B * K);
    // both matrices of one type, the activation rows fit in LDS: the launch whose groups own whole Q8_1 blocks (ffn.hip; no counters used)
    if (type_gate == type_up && B * (K + K / 4) <= 40960 && N / 32 < 0x7fffffff)
        return launch_gate_up_blk(s, type_gate, w_gate, w_up, aq, ads, K, B, gate, up, out_stride, act_out, N);
    const int64_t per = N / 8;   // groups per matrix: 4 waves x 2 rows
    MI355_REQUIRE(2 * per < 0x7fffffff, "ffn_gate_up_swiglu: too many rows for one launch");
    gemv_batch b;
    b.n = 2;
    for (int i = 0; i < 4; i++) {
        const int j = i & 1;
        b.it[i].W = (const uint8_t *)(j ? w_up : w_gate);
        b.it[i].dst = j ? up : gate;
        b.it[i].residual = nullptr;
        b.it[i].N = N;
        b.it[i].dst_stride = out_stride;
        b.it[i].type = j ? type_up : type_gate;
        b.it[i].first_group = (int)(j * per);
        b.it[i].epi = EPI_STORE;
        b.it[i].nb1 = b.it[i].nb2 = 0;
    }
    gemv_tail t;
    t.counters = counters; t.x2 = up; t.n = (int)N;
    t.act_q = (int8_t *)act_out;
    t.act_s = (act_ds *)(t.act_q + B * N);
    const dim3 grid((unsigned)(2 * per));
    const size_t lds = act_lds_bytes((int)B, K, 2 * per);
    switch (B) {
        case 1:
            if (lds) MI355_LAUNCH((k_gemv_gate_up<1, true>), grid, dim3(256), lds, s, b, aq, ads, (int)K, t);
            else MI355_LAUNCH((k_gemv_gate_up<1, false>), grid, dim3(256), 0, s, b, aq, ads, (int)K, t);
            break;
        case 2:
            if (lds) MI355_LAUNCH((k_gemv_gate_up<2, true>), grid, dim3(256), lds, s, b, aq, ads, (int)K, t);
            else MI355_LAUNCH((k_gemv_gate_up<2, false>), grid, dim3(256), 0, s, b, aq, ads, (int)K, t);
            break;
        case 3:
            if (lds) MI355_LAUNCH((k_gemv_gate_up<3, true>), grid, dim3(256), lds, s, b, aq, ads, (int)K, t);
            else MI355_LAUNCH((k_gemv_gate_up<3, false>), grid, dim3(256), 0, s, b, aq, ads, (int)K, t);
            break;
        default:
            if (lds) MI355_LAUNCH((k_gemv_gate_up<4, true>), grid, dim3(256), lds, s, b, aq, ads, (int)K, t);
            else MI355_LAUNCH((k_gemv_gate_up<4, false>), grid, dim3(256), 0, s, b, aq, ads, (int)K, t);
            break;
    }
    return launch_status("k_gemv_gate_up");
}

// act: split layout of nb1*T quantized rows of b.  dst [N, n_used, T] contiguous.
int mi355_mul_mat_id_vec(void *stream, int type, const void *as, const void *act, const int32_t *ids, int64_t ids_stride,
                         float *dst, int64_t N, int64_t K, int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T) {
    MI355_REQUIRE(is_weight_type(type), "mul_mat_id: unsupported weight type %d", type);
    MI355_REQUIRE(N > 0 && K > 0 && K < (int64_t(1) << 30) && n_expert > 0 && n_used > 0 && nb1 > 0 && T > 0, "mul_mat_id: bad shape");
    MI355_REQUIRE(K % type_block_elems(type) == 0, "mul_mat_id: K=%lld is not a multiple of the block size", (long long)K);
    MI355_REQUIRE(n_used * T <= 65535, "mul_mat_id: too many expert slots for one launch");
    const row_layout L = make_row_layout(type, K);
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + nb1 * T * K);
    if (!layout_loadable(as)) {
        const dim3 ugrid((unsigned)N, (unsigned)(n_used * T));
#define MI355_ID_UNALIGNED_LAUNCH(TY) MI355_LAUNCH(k_gemv_id_unaligned<TY>, ugrid, dim3(64), 0, s, (const uint8_t *)as, aq, ads, ids, ids_stride, dst, N, K, n_expert, n_used, nb1, L);
        MI355_WEIGHT_TYPE_SWITCH(type, MI355_ID_UNALIGNED_LAUNCH)
#undef MI355_ID_UNALIGNED_LAUNCH
        return launch_status("k_gemv_id_unaligned");
    }
    const int rpw = pick_rpw(N * n_used) > 2 ? 2 : pick_rpw(N * n_used);
    const dim3 grid((unsigned)((N + 4 * rpw - 1) / (4 * rpw)), (unsigned)(n_used * T));
    // an activation row of the split layout is 16-byte aligned inside the workspace when K % 64 == 0 (levels and scales)
    const size_t lds = K % 64 == 0 ? act_lds_bytes(1, K, (int64_t)grid.x * grid.y) : 0;
#define MI355_ID_LAUNCH(TY)                                                                                           \
    if (lds && rpw == 1) MI355_LAUNCH((k_gemv_id<TY, 1, true>), grid, dim3(256), lds, s, (const uint8_t *)as, aq, ads, ids, ids_stride, dst, N, (int)K, n_expert, n_used, nb1); \
    else if (lds) MI355_LAUNCH((k_gemv_id<TY, 2, true>), grid, dim3(256), lds, s, (const uint8_t *)as, aq, ads, ids, ids_stride, dst, N, (int)K, n_expert, n_used, nb1); \
    else if (rpw == 1) MI355_LAUNCH((k_gemv_id<TY, 1, false>), grid, dim3(256), 0, s, (const uint8_t *)as, aq, ads, ids, ids_stride, dst, N, (int)K, n_expert, n_used, nb1); \
    else MI355_LAUNCH((k_gemv_id<TY, 2, false>), grid, dim3(256), 0, s, (const uint8_t *)as, aq, ads, ids, ids_stride, dst, N, (int)K, n_expert, n_used, nb1);
    MI355_WEIGHT_TYPE_SWITCH(type, MI355_ID_LAUNCH)
#undef MI355_ID_LAUNCH
    return launch_status("k_gemv_id");
}

int mi355_moe_gate_up_swiglu_supported(int type, const void *as_gate, const void *as_up, int64_t N, int64_t K) {
    if (!is_weight_type(type) || N <= 0 || N % 32 != 0 || N / 32 >= 0x7fffffff || K <= 0 || K > 32768 || K % 64 != 0 || K % type_block_elems(type) != 0) return 0;
    const row_layout L = make_row_layout(type, K);
    return layout_aligned(as_gate, L) && layout_aligned(as_up, L) ? 1 : 0;
}

int mi355_moe_gate_up_swiglu(void *stream, int type, const void *as_gate, const void *as_up, const void *act, const int32_t *ids, int64_t ids_stride,
                             float *gate, float *up, void *act_out, int64_t N, int64_t K, int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T) {
    MI355_REQUIRE(is_weight_type(type), "moe_gate_up_swiglu: unsupported weight type %d", type);
    MI355_REQUIRE(N > 0 && N % 32 == 0 && N / 32 < 0x7fffffff && K > 0 && K <= 32768 && n_expert > 0 && n_used > 0 && nb1 > 0 && T > 0,
                  "moe_gate_up_swiglu: bad shape (N must be a multiple of 32, K at most 32768)");
    MI355_REQUIRE(K % type_block_elems(type) == 0 && K % 64 == 0, "moe_gate_up_swiglu: K=%lld must be a multiple of the block size and of 64", (long long)K);
    MI355_REQUIRE(n_used * T <= 65535, "moe_gate_up_swiglu: too many expert slots for one launch");
    MI355_REQUIRE(ids != nullptr && gate != nullptr && up != nullptr && ((uintptr_t)act & 15) == 0 && ((uintptr_t)act_out & 15) == 0,
                  "moe_gate_up_swiglu: misaligned or missing operands");
    const row_layout L = make_row_layout(type, K);
    MI355_REQUIRE(layout_aligned(as_gate, L) && layout_aligned(as_up, L), "moe_gate_up_swiglu: expert rows must be 16-byte aligned");
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + nb1 * T * K);
    return launch_gate_up_blk_id((hipStream_t)stream, type, as_gate, as_up, aq, ads, ids, ids_stride, K, gate, up, act_out, N, n_expert, n_used, nb1, T);
}

int mi355_block_dots_q8_1(void *stream, int type, const void *W, const void *a, int32_t *out, int64_t N, int64_t K) {
    int rc = check_gemv_args("block_dots", type, W, N, K, N);
    if (rc != MI355_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)a;
    const act_ds *ads = (const act_ds *)(aq + K);
    const dim3 grid((unsigned)N);
#define MI355_BLOCK_DOTS_LAUNCH(TY) MI355_LAUNCH(k_block_dots<TY>, grid, dim3(64), 0, s, (const uint8_t *)W, aq, ads, out, N, (int)K);
    MI355_WEIGHT_TYPE_SWITCH(type, MI355_BLOCK_DOTS_LAUNCH)
#undef MI355_BLOCK_DOTS_LAUNCH
    return launch_status("k_block_dots");
}

}  // extern "C"
