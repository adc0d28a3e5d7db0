// Sums of partial results: a product cut along K leaves n_slices slabs, added in ascending order.
#pragma once
#include "common.hpp"

namespace mi355 {

// Four neighbouring elements of every slab, `stride` floats apart.  All slabs are requested before the first is waited for (a loop over their number waits for each in turn,
// a trip to memory per slab): SL = their number where that is 2 .. 4, 0 = any, four at a time.
template <int SL> struct slab_sum {
    static constexpr int AHEAD = SL ? SL : 4;
    f32x4 t[AHEAD];
    __device__ __forceinline__ void request(const float *__restrict__ part, int64_t stride, int n_slices) {
#pragma unroll
        for (int j = 0; j < AHEAD; j++) t[j] = *(const f32x4 *)(part + (SL || j < n_slices ? j : 0) * stride);
    }
    __device__ __forceinline__ f32x4 sum(const float *__restrict__ part, int64_t stride, int n_slices) {
        f32x4 acc = t[0];
#pragma unroll
        for (int j = 1; j < AHEAD; j++) {
            if (!SL && j >= n_slices) break;   // uniform
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = add_rn(acc[i], t[j][i]);
        }
        if constexpr (SL == 0) {
            for (int s0 = 4; s0 < n_slices; s0 += 4) {
#pragma unroll
                for (int j = 0; j < 4; j++) t[j] = *(const f32x4 *)(part + (s0 + j < n_slices ? s0 + j : s0) * stride);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (s0 + j >= n_slices) break;   // uniform
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[i] = add_rn(acc[i], t[j][i]);
                }
            }
        }
        return acc;
    }
};
// LAUNCH(SL) for n slices
#define MI355_SLAB_SWITCH(n, LAUNCH) \
    switch (n) {                     \
        case 2: LAUNCH(2); break;    \
        case 3: LAUNCH(3); break;    \
        case 4: LAUNCH(4); break;    \
        default: LAUNCH(0); break;   \
    }

}  // namespace mi355
