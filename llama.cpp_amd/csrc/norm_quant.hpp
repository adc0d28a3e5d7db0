// RMS_NORM -> MUL(weight) [-> Q8_1 | Q8_K] of one row by one 256-thread group (ggml_compute_forward_rms_norm_f32,
// ggml/src/ggml-cpu/ggml-cpu.c:6741-6805; quantize_row_q8_1_ref, ggml/src/ggml-quants.c:220-253).  A device function, so that
// a launch which finishes rows can also normalise them; every rounding of the reduction is spelled out, so all callers give
// the same bits.
#pragma once
#include "common.hpp"
#include "q8k.hpp"
#include "tiles.hpp"

namespace mi355 {

// Q8_1 of the 4 values held by each of 8 neighbouring lanes (one 32-element block); writes the
// split activation layout.  Mirrors k_quantize_q8_1 (quantize.hip) instruction for instruction.
__device__ __forceinline__ void quantize_block_lane(const f32x4 &v, bool live, int8_t *__restrict__ qplane, act_ds *__restrict__ ds,
                                                    int64_t row, int64_t k, int64_t e0) {
    const float amax = lanes_max<8>(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    float d, id;
    q8_scale(amax, d, id);
    int q[4];
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        q[i] = q8_level(v[i], id);
        sum += q[i];
    }
    sum = lanes_sum_i<8>(sum);
    if (!live) return;
    const u32 packed = (u32)(q[0] & 0xFF) | ((u32)(q[1] & 0xFF) << 8) | ((u32)(q[2] & 0xFF) << 16) | ((u32)(q[3] & 0xFF) << 24);
    *(u32 *)(qplane + row * k + e0) = packed;
    if (((e0 >> 2) & 7) == 0) {
        act_ds o;
        o.d = half_bits_to_float(float_to_half_bits(d));
        o.sum = sum;
        ds[row * (k >> 5) + (e0 >> 5)] = o;
    }
}

// Q8_1 of one value per lane over aligned groups of 32 lanes (quantize_row_q8_1_ref, ggml-quants.c:220-253); e = index of the
// lane's element in the row.  COH: the block is stored with device scope (four levels per store, the {d, sum} pair as one
// 8-byte store), for rows that other groups of the same launch read after a grid-wide step.
template <bool COH = false>
__device__ __forceinline__ void quantize_lane32(float v, int8_t *__restrict__ qrow, act_ds *__restrict__ srow, int64_t e) {
    const float amax = lanes_max<32>(fabsf(v));
    float d, id;
    q8_scale(amax, d, id);
    const int q = q8_level(v, id);
    const int sum = lanes_sum_i<32>(q);
    act_ds o;
    o.d = half_bits_to_float(float_to_half_bits(d));
    o.sum = sum;
    if constexpr (COH) {
        u32 packed = (u32)(q & 0xFF);
        packed |= ((u32)__shfl_down(q, 1, 64) & 0xFFu) << 8;
        packed |= ((u32)__shfl_down(q, 2, 64) & 0xFFu) << 16;
        packed |= ((u32)__shfl_down(q, 3, 64) & 0xFFu) << 24;
        if ((e & 3) == 0) __hip_atomic_store((u32 *)(qrow + e), packed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((e & 31) == 0) {
            const unsigned long long bits = (unsigned long long)__builtin_bit_cast(u32, o.d) | ((unsigned long long)(u32)o.sum << 32);
            __hip_atomic_store((unsigned long long *)(srow + (e >> 5)), bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    } else {
        qrow[e] = (int8_t)q;
        if ((e & 31) == 0) srow[e >> 5] = o;
    }
}

// Sum of squares of the thread's pieces -> the row's 1 / rms in every thread.  The first 256 threads' sums count (sh: 4 floats of LDS; the caller places a barrier
// between two calls that share it).  Contains exactly one group barrier, which further waves of a larger group must match with a barrier of their own.
template <int NV>
__device__ __forceinline__ float rms_norm_scale(const f32x4 (&v)[NV], int64_t k, float eps, float *sh) {
    const int tid = threadIdx.x;
    float ss = 0.0f;
#pragma unroll
    for (int it = 0; it < NV; it++)
#pragma unroll
        for (int i = 0; i < 4; i++) ss = __builtin_fmaf(v[it][i], v[it][i], ss);
    ss = wave_sum_dpp(ss);
    if ((tid & 63) == 0 && tid < 256) sh[tid >> 6] = ss;
    __syncthreads();
    ss = add_rn(add_rn(add_rn(sh[0], sh[1]), sh[2]), sh[3]);
    return 1.0f / sqrtf(add_rn(ss / (float)k, eps));
}

// Q8_1 of eight neighbouring values per lane over aligned groups of four lanes into a row's LDS copy (levels, then {d, sum} of every block); e0 = the lane's first element.
// Same levels and scales as quantize_block_lane: of the work per block only the maximum and the sum are more than one lane's, and a third of the instructions per element
// remain of four lanes doing what eight did twice.
__device__ __forceinline__ void quantize_block_lane8(const f32x4 (&v)[2], int8_t *__restrict__ qrow, act_ds *__restrict__ srow, int e0) {
    float amax = fmaxf(fabsf(v[0][0]), fabsf(v[1][0]));
#pragma unroll
    for (int i = 1; i < 4; i++) amax = fmaxf(amax, fmaxf(fabsf(v[0][i]), fabsf(v[1][i])));
    amax = lanes_max<4>(amax);
    float d, id;
    q8_scale(amax, d, id);
    u32x2 packed;
    int sum = 0;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        u32 q[4];
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = (u32)q8_level(v[j][i], id);
        packed[j] = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u) | __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);   // the low bytes in order
        sum = dot4((int)packed[j], 0x01010101, sum);
    }
    sum = lanes_sum_i<4>(sum);
    *(u32x2 *)(qrow + e0) = packed;
    if ((e0 & 31) == 0) {
        act_ds o;
        o.d = half_bits_to_float(float_to_half_bits(d));
        o.sum = sum;
        srow[e0 >> 5] = o;
    }
}

// RMS_NORM -> MUL -> Q8_1 of one row of at most 4096 elements (a multiple of 1024) into a group's LDS copy, in two parts: request() ahead of the group's
// first weight loads - a wave's loads return in the order of their issue - and finish() behind them.  Same bits as rms_norm_quant_row: the first four waves form its
// sum in its order, then every thread quantizes its share, eight elements at a time.  WAVES: 4 or 8.
template <int WAVES>
struct norm_row {
    static constexpr int NP = 8 / WAVES;
    f32x4 v[4], own[NP][2], w[NP][2];
    static __device__ __forceinline__ int element(int it) { return (it * 256 + (int)(threadIdx.x & 255)) * 4; }
    static __device__ __forceinline__ int first(int p) { return (p * 64 * WAVES + (int)threadIdx.x) * 8; }
    __device__ __forceinline__ void request(const float *__restrict__ x, const float *__restrict__ nw, int K) {
        // pieces past the end repeat others, and nothing uses them: a branch around a load would let the compiler move it to where its value is needed
#pragma unroll
        for (int it = 0; it < 4; it++) v[it] = *(const f32x4 *)(x + (element(it) < K ? element(it) : element(0)));
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int e0 = first(p), at = e0 < K ? e0 : 0;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                own[p][j] = *(const f32x4 *)(x + at + 4 * j);
                w[p][j] = *(const f32x4 *)(nw + at + 4 * j);
            }
        }
    }
    __device__ __forceinline__ void finish(uint8_t *s_act, int K, float eps, float *sh) {
#pragma unroll
        for (int it = 1; it < 4; it++)
            if (it * 1024 >= K) v[it] = f32x4{0.f, 0.f, 0.f, 0.f};   // uniform
        const float scale = rms_norm_scale<4>(v, K, eps, sh);   // (further waves repeat the first four's sums, which are not used: a branch, see request())
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int e0 = first(p);
            if (e0 >= K) return;   // uniform over the wave
            f32x4 o[2];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    o[j][i] = own[p][j][i] * scale;
                    o[j][i] = o[j][i] * w[p][j][i];
                }
            quantize_block_lane8(o, (int8_t *)s_act, (act_ds *)(s_act + K), e0);
        }
    }
};

// Four elements of the row from e0 on, normalised (a wave's lanes hold 256 neighbouring ones) -> y row and activation, as rms_norm_quant_row
template <int FMT>
__device__ __forceinline__ f32x4 norm_piece(const f32x4 &v, const f32x4 &w, bool weighted, float scale, float *__restrict__ yr, void *__restrict__ act, int64_t row,
                                            int64_t k, int64_t nrows, int64_t e0) {
    const bool live = e0 < k;
    int8_t *qplane = (int8_t *)act;
    f32x4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = v[i] * scale;
    if (weighted && live) {
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = o[i] * w[i];
    }
    if (yr && live) *(f32x4 *)(yr + e0) = o;
    if constexpr (FMT == 2) {
        if (act && live) q8k_quantize_wave_tiled(o, threadIdx.x & 63, (uint8_t *)act, k, nrows, row, e0 >> 8);   // whole wave: k is a multiple of 256
    } else if constexpr (FMT == 1) {
        if (act && live) {   // whole wave: k is a multiple of 256
            const int64_t nsb = k >> 8, sb = e0 >> 8;
            float *d8 = (float *)(qplane + q8k_d_offset(k, nrows));
            _Float16 *bs = (_Float16 *)(qplane + q8k_bs_offset(k, nrows));
            q8k_quantize_wave(o, threadIdx.x & 63, qplane + row * k + sb * QKK, d8 + row * nsb + sb, bs + (row * nsb + sb) * 16);
        }
    } else {
        if (act) quantize_block_lane(o, live, qplane, (act_ds *)(qplane + nrows * k), row, k, e0);
    }
    return o;
}

// One row by 1024 threads, for launches of a few rows: such a launch is one dependent chain per wave, some 2 ns per instruction, and with sixteen waves a thread of a
// row of 4096 quantizes four elements instead of sixteen.  Same bits as rms_norm_quant_row: the first four waves form its sum in its order.  NV: pieces of a 256-thread
// group (k <= 1024 * NV).  sh: 4 floats of LDS.
template <int NV, int FMT>
__device__ __forceinline__ void rms_norm_quant_row_wide(const float *__restrict__ xr, const float *__restrict__ w, float *__restrict__ yr, void *__restrict__ act, int64_t row,
                                                        int64_t k, int64_t nrows, float eps, float *sh) {
    constexpr int NP = NV / 4;
    const int tid = threadIdx.x;
    // Everything is requested before anything is waited for; pieces past the end repeat the first one, and nothing uses them (a branch around each load made three trips to memory of
    // one: one row of 4096 2.43 us, now 2.29; to a Q8_K image 3.2, now 2.7).
    f32x4 own[NP], ww[NP];
    const float *wr = w ? w : xr;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int64_t e0 = ((int64_t)p * 1024 + tid) * 4, at = e0 < k ? e0 : 0;
        own[p] = *(const f32x4 *)(xr + at);
        ww[p] = *(const f32x4 *)(wr + at);
    }
    const float kf = (float)k;
    asm volatile("" ::"s"(eps), "s"(kf), "s"(nrows));   // (arguments beyond the preloaded ones)
    if (__builtin_amdgcn_readfirstlane(tid >> 8) == 0) {
        f32x4 v[NV];
#pragma unroll
        for (int it = 0; it < NV; it++) {
            const int64_t e0 = ((int64_t)it * 256 + tid) * 4;
            v[it] = *(const f32x4 *)(xr + (e0 < k ? e0 : 0));
        }
        float ss = 0.0f;
#pragma unroll
        for (int it = 0; it < NV; it++) {
            const bool live = ((int64_t)it * 256 + tid) * 4 < k;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float t = live ? v[it][i] : 0.0f;
                ss = __builtin_fmaf(t, t, ss);
            }
        }
        ss = wave_sum_dpp(ss);
        if ((tid & 63) == 0) sh[tid >> 6] = ss;
    }
    __syncthreads();
    const float total = add_rn(add_rn(add_rn(sh[0], sh[1]), sh[2]), sh[3]);
    const float scale = 1.0f / sqrtf(add_rn(total / kf, eps));
#pragma unroll
    for (int p = 0; p < NP; p++) norm_piece<FMT>(own[p], ww[p], w != nullptr, scale, yr, act, row, k, nrows, ((int64_t)p * 1024 + tid) * 4);
}

// One row: xr -> y row (optional) and row `row` of the activation workspace `act` (optional), which holds nrows rows of k.
// Each thread keeps its NV float4 of the row in registers (k <= 1024 * NV).  COH: the row was written by other groups of the
// same launch with device-scope stores and is read with device-scope loads.  sh: 4 floats of LDS; the caller places a
// barrier between two calls that share it.
// FMT: activation format written to `act`: 0 Q8_1 (split layout), 1 per-super-block (q8k.hpp), 2 the same as tile images (tiles.hpp)
// Called by the first 256 threads of a group; contains exactly one group barrier, which further waves of a larger group must
// match with a barrier of their own.
// keep: where the caller wants the thread's NV pieces of the normalised row (registers), or null
template <int NV, int FMT, bool COH>
__device__ __forceinline__ void rms_norm_quant_row(const float *__restrict__ xr, const float *__restrict__ w, float *__restrict__ yr,
                                                   void *__restrict__ act, int64_t row, int64_t k, int64_t nrows, float eps, float *sh,
                                                   f32x4 *keep = nullptr) {
    const int tid = threadIdx.x;
    f32x4 v[NV], ww[NV];
    // the weight does not depend on the reduction: fetch it together with the row, one memory round trip instead of two; pieces past the end repeat the first one and are not used (a
    // branch around every load makes a trip of each)
    const float *wr = w ? w : xr;
#pragma unroll
    for (int it = 0; it < NV; it++) {
        const int64_t e0 = ((int64_t)it * 256 + tid) * 4, at = e0 < k ? e0 : 0;
        if constexpr (COH) {
#pragma unroll
            for (int i = 0; i < 4; i++) v[it][i] = __hip_atomic_load(xr + at + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            v[it] = *(const f32x4 *)(xr + at);
        }
    }
#pragma unroll
    for (int it = 0; it < NV; it++) {
        const int64_t e0 = ((int64_t)it * 256 + tid) * 4;
        ww[it] = *(const f32x4 *)(wr + (e0 < k ? e0 : 0));
    }
#pragma unroll
    for (int it = 0; it < NV; it++)
        if (((int64_t)it * 256 + tid) * 4 >= k) v[it] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float scale = rms_norm_scale<NV>(v, k, eps, sh);
#pragma unroll
    for (int it = 0; it < NV; it++) {
        const f32x4 o = norm_piece<FMT>(v[it], ww[it], w != nullptr, scale, yr, act, row, k, nrows, ((int64_t)it * 256 + tid) * 4);
        if (keep) keep[it] = o;
    }
}

}  // namespace mi355
