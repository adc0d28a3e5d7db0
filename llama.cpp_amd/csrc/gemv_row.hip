// One activation row against one matrix (wo, ffn_down of a decoded token): dst[n] = W[n] . x (+ residual[n]), a wave per weight row.
//
// Such a launch is over when its slowest chain is: its groups are mostly resident at once, and a wave of k_gemv_q walked a row of 14336 in four steps, each a round trip for the
// weights and, behind them, for the activation.  Here a group copies the activation to LDS first (a wave's loads return in the order of their issue), every wave has
// gr_steps of its row on their way from the start - the 33 MB of a 4096 x 14336 Q4_K matrix all at once, 130 KB per compute unit - and the residual is requested ahead of everything.
// 8B shapes in a chain of launches, us: wo 4.6 -> 3.8, ffn_down Q4_K 10.9 -> 8.0, Q6_K 11.4 -> 10.2 (8.2, 10.8 before the loads of a step were kept together; 8192 x 28672 Q4_K 25.3 -> 24.1; other figures: gemv_row.hpp).
// Sums as in gemv_body: same lane-to-chunk mapping, same order of steps, same wave reduction.
#include "common.hpp"
#include "qdot.hpp"
#include "gemv_row.hpp"

namespace mi355 {

extern __shared__ __attribute__((aligned(16))) uint8_t s_gr[];

// steps in flight: four, two of the types whose chunks take the most registers or the most loads (4096 x 14336, four / two: Q5_K 14.3 / 10.9 us, IQ4_XS 10.6 / 9.2, Q6_K 10.8 / 10.9 alone
// and 48.5 / 48.0 for the layer)
template <int TYPE> constexpr int gr_steps() { return TYPE == MI355_Q6_K || TYPE == MI355_Q5_K || TYPE == MI355_IQ4_XS ? 2 : 4; }

// Waves per SIMD the registers are to leave room for.  IQ4_XS would take 67 of them, three past eight waves: 8192 rows are 1024 groups, four to every compute unit, of which three fit then
// and the last ones run alone.  us, k_gemv_q / this with 67 / with 64 registers: 8192 x 4096 6.6 / 6.4 / 5.9, x 6144 8.9 / 8.9 / 8.5, x 14336 16.1 / 16.6 / 15.2.  (IQ4_NL, 68 registers
// with four steps: 64 of them spill, 8192 x 14336 12.8 % slower; as it is 8192 x 6144 is the one size of all types found slower than k_gemv_q beyond the noise, by 1 %.)
template <int TYPE> constexpr int gr_min_waves() { return TYPE == MI355_IQ4_XS ? 8 : 1; }

template <int TYPE, int STEPS, int WAVES, int KMAX>
__global__ void __launch_bounds__(64 * WAVES, gr_min_waves<TYPE>()) k_gemv_row(const uint8_t *__restrict__ W, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, float *dst,
                                                         const float *residual, int N, int K) {   // residual may be dst: a row's is read by the wave that stores it
    typedef wq<TYPE> T;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = (int)blockIdx.x * WAVES + wave, at = row < N ? row : N - 1;   // rows past the end repeat the last one and are not stored
    const row_layout L = make_row_layout(TYPE, K);
    const int nchunks = K / T::CHUNK;
    const uint8_t *wrow = W + (int64_t)at * L.row_bytes;

    const float res = *(residual ? residual + at : (const float *)ads);   // (without one some word of the activation, not used)
    act_copy<1, 64 * WAVES, KMAX, true> copy;
    copy.request(aq, ads, K);
    __builtin_amdgcn_sched_barrier(0);
    typedef late_chunk<TYPE> G;
    typename G::raw w[STEPS];
#pragma unroll
    for (int p = 0; p < STEPS; p++) {
        const int c = p * 64 + lane;
        w[p] = G::load(wrow, L, c < nchunks ? c : nchunks - 1);
        if constexpr (G::ORDERED) __builtin_amdgcn_sched_barrier(0);   // step by step, here and below: a step must not wait for pieces of a later one
    }
    copy.commit(s_gr, aq, ads, K);
    __syncthreads();
    const int8_t *s_q = (const int8_t *)s_gr;
    const act_ds *s_ds = (const act_ds *)(s_gr + K);
    float acc = 0.0f;
    // rounds of STEPS steps; a step's registers take the one STEPS further on without a condition (past the end the last chunk again): at the join of two paths the
    // compiler knows the smaller number of loads in flight only, and waits for more than it needs
    int c0 = 0;
    for (; c0 + 64 * STEPS < nchunks; c0 += 64 * STEPS) {
#pragma unroll
        for (int p = 0; p < STEPS; p++) {
            const int c = c0 + p * 64 + lane, next = c + 64 * STEPS;
            const typename T::act A = T::load_a(s_q, s_ds, c);
            const typename T::chunk now = G::decode(w[p], c);
            acc = T::accumulate(acc, now, A, T::dots(now, A));
            w[p] = G::load(wrow, L, next < nchunks ? next : nchunks - 1);
            if constexpr (G::ORDERED) __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int p = 0; p < STEPS; p++) {
        const int c = c0 + p * 64 + lane;
        if (c0 + p * 64 >= nchunks) break;   // uniform
        const typename T::act A = T::load_a(s_q, s_ds, c < nchunks ? c : nchunks - 1);
        const typename T::chunk now = G::decode(w[p], c);
        const float sum = T::accumulate(acc, now, A, T::dots(now, A));
        acc = c < nchunks ? sum : acc;
    }
    const float s = wave_sum_dpp(acc);
    if (lane == 0 && row < N) dst[row] = residual ? s + res : s;
}

template <int TYPE, int STEPS, int KMAX>
static void launch_steps(hipStream_t s, const void *W, const int8_t *aq, const act_ds *ads, float *dst, const float *residual, int64_t N, int64_t K) {
    const size_t lds = (size_t)(K + K / 4);
    if (N <= 2048) MI355_LAUNCH((k_gemv_row<TYPE, STEPS, 4, KMAX>), dim3((unsigned)((N + 3) / 4)), dim3(256), lds, s, (const uint8_t *)W, aq, ads, dst, residual, (int)N, (int)K);
    else MI355_LAUNCH((k_gemv_row<TYPE, STEPS, 8, KMAX>), dim3((unsigned)((N + 7) / 8)), dim3(512), lds, s, (const uint8_t *)W, aq, ads, dst, residual, (int)N, (int)K);
}

int launch_gemv_row(hipStream_t s, int type, const void *W, const int8_t *aq, const act_ds *ads, float *dst, const float *residual, int64_t N, int64_t K) {
#define MI355_GR_LAUNCH(TY)                                                                                             \
    if (K / wq<TY>::CHUNK <= 64) launch_steps<TY, 1, 4096>(s, W, aq, ads, dst, residual, N, K);                         \
    else if (K / wq<TY>::CHUNK <= 128) launch_steps<TY, 2, 8192>(s, W, aq, ads, dst, residual, N, K);                   \
    else if (K <= 16384) launch_steps<TY, gr_steps<TY>(), 16384>(s, W, aq, ads, dst, residual, N, K);                   \
    else launch_steps<TY, gr_steps<TY>(), 32768>(s, W, aq, ads, dst, residual, N, K);
    MI355_WEIGHT_TYPE_SWITCH(type, MI355_GR_LAUNCH)
#undef MI355_GR_LAUNCH
    return launch_status("k_gemv_row");
}

}  // namespace mi355
