// MUL_MAT of one to three f32 activation rows in ONE launch: dst[b][n] = sum_k W[n][k] * x[b][k], x quantized to Q8_1 on the way.
//
// mi355_quantize_act followed by k_gemv_q is two dependent launches of 2.2 and 4.2 us (4096 x 4096 Q4_K), each with its own host time and
// the gap between them.  Here every group quantizes the rows for itself, straight into the LDS copy its waves read the levels from, while
// its first weight loads are on their way: groups x 4 K B more bytes out of L2, one launch less.
#include "common.hpp"
#include "qdot.hpp"
#include "norm_quant.hpp"

namespace mi355 {

constexpr int GF_WAVES = 8;   // per group: half the groups, half the quantization work of four

extern __shared__ __attribute__((aligned(16))) uint8_t s_gf[];

// Same arithmetic, lane-to-chunk mapping and order of sums as quantize_row_q8_1_ref's launch and gemv_body: the bytes of the result are theirs.
template <int TYPE, int NCOLS, int RPW>
__global__ void __launch_bounds__(GF_WAVES * 64) k_gemv_f32(const uint8_t *__restrict__ W, const float *__restrict__ x, float *__restrict__ dst, int64_t N, int K,
                                                           int64_t x_stride, int64_t dst_stride) {
    typedef wq<TYPE> T;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = ((int64_t)blockIdx.x * GF_WAVES + wave) * RPW;
    const row_layout L = make_row_layout(TYPE, K);
    const int nchunks = K / T::CHUNK, nblk = K >> 5;

    int8_t *s_q = (int8_t *)s_gf;
    act_ds *s_ds = (act_ds *)(s_gf + NCOLS * K);
    constexpr int STEP = GF_WAVES * 64 * 4, PIECES = 2;
    f32x4 v[NCOLS][PIECES];   // 4096 elements of every row in flight
    auto request = [&](int k0) {
#pragma unroll
        for (int col = 0; col < NCOLS; col++)
#pragma unroll
            for (int i = 0; i < PIECES; i++) {
                const int k = k0 + i * STEP + (int)threadIdx.x * 4;
                v[col][i] = *(const f32x4 *)(x + col * x_stride + (k < K ? k : K - 4));
            }
    };
    // x first, the first step's weights behind it: a wave's loads return in the order of their issue, and the rows are quantized while the weights arrive
    request(0);
    __builtin_amdgcn_sched_barrier(0);
    const uint8_t *rows[RPW];
    typename T::chunk w_first[RPW];
#pragma unroll
    for (int r = 0; r < RPW; r++) {
        const int64_t row = row0 + r < N ? row0 + r : N - 1;   // rows past the end repeat the last one and are not stored
        rows[r] = W + row * L.row_bytes;
        w_first[r] = T::load_w(rows[r], L, lane < nchunks ? lane : nchunks - 1);
    }
    auto quantize = [&](int k0) {
#pragma unroll
        for (int col = 0; col < NCOLS; col++)
#pragma unroll
            for (int i = 0; i < PIECES; i++) {
                const int k = k0 + i * STEP + (int)threadIdx.x * 4;
                quantize_block_lane(v[col][i], k < K, s_q, s_ds, col, K, k);
            }
    };
    quantize(0);
    for (int k0 = PIECES * STEP; k0 < K; k0 += PIECES * STEP) {
        request(k0);
        quantize(k0);
    }
    __syncthreads();
    if (row0 >= N) return;   // whole wave

    float acc[RPW][NCOLS];
#pragma unroll
    for (int r = 0; r < RPW; r++)
#pragma unroll
        for (int c = 0; c < NCOLS; c++) acc[r][c] = 0.0f;
    for (int c0 = 0; c0 < nchunks; c0 += 64) {
        const int c = c0 + lane;
        if (c < nchunks) {
            typename T::chunk w[RPW];
#pragma unroll
            for (int r = 0; r < RPW; r++) w[r] = c0 == 0 ? w_first[r] : T::load_w(rows[r], L, c);
#pragma unroll
            for (int col = 0; col < NCOLS; col++) {
                const typename T::act A = T::load_a(s_q + col * K, s_ds + col * nblk, c);
#pragma unroll
                for (int r = 0; r < RPW; r++) acc[r][col] = T::accumulate(acc[r][col], w[r], A, T::dots(w[r], A));
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RPW; r++)
#pragma unroll
        for (int c = 0; c < NCOLS; c++) {
            const float s = wave_sum_dpp(acc[r][c]);
            if (lane == 0 && row0 + r < N) dst[c * dst_stride + row0 + r] = s;
        }
}

// rows per wave: two, so that 4096 weight rows are one group per compute unit; one where even that leaves units idle
static int gf_rpw(int64_t N) { return N <= 2048 ? 1 : 2; }

// Where one launch is the quicker form.  Device time of the two launches / of this one, us, in a graph of twenty products:
//   4096 x 4096, 1 row: Q4_K 5.6 / 3.8, Q4_0 5.6 / 4.5, Q8_0 5.5 / 3.7, Q6_K 6.3 / 5.6; 3 rows: Q4_K 7.8 / 6.1, Q8_0 7.2 / 5.7
//   1494 x 1280, 1 row: 4.2 .. 4.5 / 2.8 .. 3.2;  14336 x 4096, 1 row: Q4_K 7.7 / 7.4, Q8_0 12.8 / 10.7, Q6_K 11.2 / 11.4
// The quantization is paid once per group: from some four groups of 4096 elements per compute unit on (28672 x 8192: 22.8 / 22.5, 32768 x 2048
// 11.1 / 11.2) and, for two or three rows, from the second group per unit on (8882 x 1056 Q4_0, 2 rows: 6.2 / 6.9) it costs what the
// launch did.  Long rows are longer chains per wave here, with half of k_gemv_q's waves (4096 x 14336 Q4_0: 9.6 / 10.9).
// Inside that line the device loses where a few units get a third group or two or three rows meet the types with the most arithmetic per byte: 8975 x 5120, 1 row
// Q4_K 8.9 / 8.9, Q5_0 9.5 / 10.1, Q6_K 11.2 / 11.9, IQ4_XS 10.4 / 11.4, IQ4_NL 9.6 / 10.9; 2547 x 4096, 3 rows Q4_K 6.9 / 5.9, IQ4_NL 6.8 / 7.0, Q6_K 7.2 / 7.7.
// They stay: a call that is not replayed from a graph takes 13.5 us of host time with two launches and 7 with one.
static bool gf_faster(int64_t N, int64_t K, int64_t B) {
    if (B > 3 || K > 8192) return false;
    const int64_t groups = (N + GF_WAVES * gf_rpw(N) - 1) / (GF_WAVES * gf_rpw(N));
    return B == 1 ? groups * K <= 256 * 16384 : groups <= 256 && B * K <= 12288;
}

// whether any of the B rows of x and any of those of dst have a float in common
bool mul_mat_rows_overlap(const float *x, int64_t x_stride, int64_t K, const float *dst, int64_t dst_stride, int64_t N, int64_t B) {
    for (int64_t i = 0; i < B; i++)
        for (int64_t j = 0; j < B; j++) {
            const uintptr_t a = (uintptr_t)(x + i * x_stride), b = (uintptr_t)(dst + j * dst_stride);
            if (a < b + (uintptr_t)N * sizeof(float) && b < a + (uintptr_t)K * sizeof(float)) return true;
        }
    return false;
}

template <int TYPE, int NCOLS>
static void launch_gf(hipStream_t s, const void *W, const float *x, float *dst, int64_t N, int K, int64_t x_stride, int64_t dst_stride) {
    const size_t lds = (size_t)NCOLS * (K + K / 4);
    const int rpw = gf_rpw(N);
    const dim3 grid((unsigned)((N + GF_WAVES * rpw - 1) / (GF_WAVES * rpw))), block(GF_WAVES * 64);
    if (rpw == 1) MI355_LAUNCH((k_gemv_f32<TYPE, NCOLS, 1>), grid, block, lds, s, (const uint8_t *)W, x, dst, N, K, x_stride, dst_stride);
    else MI355_LAUNCH((k_gemv_f32<TYPE, NCOLS, 2>), grid, block, lds, s, (const uint8_t *)W, x, dst, N, K, x_stride, dst_stride);
}

}  // namespace mi355

using namespace mi355;

extern "C" {

int mi355_mul_mat_vec_f32_supported(int type, const void *W, int64_t N, int64_t K, int64_t B) {
    return is_weight_type(type) && N > 0 && K > 0 && B > 0 && K % type_block_elems(type) == 0 && layout_loadable(W) && gf_faster(N, K, B);
}

int mi355_mul_mat_vec_f32(void *stream, int type, const void *W, const float *x, float *dst, int64_t N, int64_t K, int64_t B, int64_t x_stride, int64_t dst_stride) {
    MI355_REQUIRE(mi355_mul_mat_vec_f32_supported(type, W, N, K, B), "mul_mat_vec_f32: type %d, N=%lld, K=%lld, B=%lld or the weight alignment is not served", type,
                  (long long)N, (long long)K, (long long)B);
    MI355_REQUIRE(x_stride >= K && x_stride % 4 == 0 && ((uintptr_t)x & 15) == 0, "mul_mat_vec_f32: x must be 16-byte aligned with a row stride that is a multiple of 4 floats");
    MI355_REQUIRE(dst_stride >= N, "mul_mat_vec_f32: dst_stride < N");
    MI355_REQUIRE(!mul_mat_rows_overlap(x, x_stride, K, dst, dst_stride, N, B), "mul_mat_vec_f32: dst overlaps x, which other groups still read when the first write");
    hipStream_t s = (hipStream_t)stream;
#define MI355_GF_LAUNCH(TY)                                                                 \
    if (B == 1) launch_gf<TY, 1>(s, W, x, dst, N, (int)K, x_stride, dst_stride);            \
    else if (B == 2) launch_gf<TY, 2>(s, W, x, dst, N, (int)K, x_stride, dst_stride);       \
    else launch_gf<TY, 3>(s, W, x, dst, N, (int)K, x_stride, dst_stride);
    MI355_WEIGHT_TYPE_SWITCH(type, MI355_GF_LAUNCH)
#undef MI355_GF_LAUNCH
    return launch_status("k_gemv_f32");
}

}  // extern "C"
