// MUL_MAT for a handful of activation rows (4 .. 32): weight-streaming kernel on the int8 matrix cores.
//
// The batch-1 kernels (gemv.hip) spend eight v_dot4 per weight block and activation row, which binds them to the vector
// ALUs from about five activation rows on; the tile kernels (mmq.hip, mmq_k.hip) are built around 64..128-row activation
// tiles and a K loop with group barriers, and a launch with one tile column is latency-bound.  Here a wave owns 32 weight
// rows and one quarter of K and never waits for another wave until the end:
//   * per step of 256 elements the wave copies its weights (32 rows), activation rows and activation scales to its own
//     part of LDS with fully coalesced 16-byte loads (a lane reads along a row; the loads of the next step are requested
//     as soon as the registers are free, before the current step is contracted), and reads them back in matrix-core
//     operand order.  Nobody else touches that part of LDS, and a wave's LDS accesses complete in program order, so no
//     barrier is involved;
//   * one v_mfma_i32_32x32x32_i8 per weight block: operand A = 16 levels of an activation row per lane (lane % 32 = row,
//     lane / 32 = half of the block), operand B = 16 levels of a weight row per lane;
//   * the result puts ONE weight row (lane % 32) and activation rows 4 (lane / 32) + 8 q + 0..3 (q = 0..3) in a lane:
//     the weight scale is one value per lane and block, the activation scales are 4 consecutive table entries per q,
//     and only the q that hold real activation rows are finished (NI = ceil(rows / 8) of them);
//   * the four K quarters of a group meet in LDS at the end and are added in a fixed order.
// Integer sums are exact, so the result differs from the batch-1 kernels' only in the order of the f32 additions.
// Activations are the Q8_1 workspace of mi355_quantize_act (ggml-cpu quantizes to Q8_0/Q8_1 for Q4_0/Q8_0 weights and to
// Q8_K for Q4_K, ggml-cpu.c:7420-7450; the NMSE bound of the product is what is checked for Q4_K).
#include "qdot.hpp"
#include "q8k.hpp"

namespace mi355 {

namespace {

// What goes through LDS per step (256 elements) and weight row: the 4-bit (Q8_0: 8-bit) plane of the levels - 128 bytes of
// nibbles for every type but Q8_0 (256, in one or two halves); Q6_K copies its 64 bytes of high bit pairs beside them.  Everything a lane needs of ITS row
// only (block scales and minima, the K-quants' 16-byte header, the fifth bits of Q5_0 / Q5_1 / Q5_K) goes straight to registers.
template <int TYPE> struct sk_traits {
    static constexpr int ROW_BYTES = TYPE == MI355_Q8_0 ? 256 : 128;
    // per-32-block types whose block is 16 bytes of nibbles, element b low and element 16 + b high in byte b
    static constexpr bool NIB32 = TYPE == MI355_Q4_0 || TYPE == MI355_IQ4_NL || TYPE == MI355_IQ4_XS || TYPE == MI355_Q4_1 || TYPE == MI355_Q5_0 ||
                                  TYPE == MI355_Q5_1;
    static constexpr bool TABLE = TYPE == MI355_IQ4_NL || TYPE == MI355_IQ4_XS;     // a nibble stands for an entry of the sixteen-value table
    static constexpr bool PAIR = TYPE == MI355_Q4_1 || TYPE == MI355_Q5_1;          // {f16 d, f16 m} per block
    static constexpr bool FIFTH32 = TYPE == MI355_Q5_0 || TYPE == MI355_Q5_1;       // one word of fifth bits per block
    static constexpr bool KQ = TYPE == MI355_Q4_K || TYPE == MI355_Q5_K;            // 16-byte header + 6-bit (scale, min) pairs
    static constexpr int STEP_BYTES = TYPE == MI355_Q8_0 ? 256 : TYPE == MI355_Q4_K ? Q4_K_BYTES : TYPE == MI355_Q5_K ? Q5_K_BYTES : 128;
    static constexpr int QS_OFF = TYPE == MI355_Q4_K ? 16 : TYPE == MI355_Q5_K ? 48 : 0;   // where the nibbles start inside a step
    // the activation's block sum enters as x = OFFSET * d * sum (levels stored with an offset) or as d * sum (block minimum)
    static constexpr float OFFSET = TYPE == MI355_Q4_0 ? -8.0f : TYPE == MI355_Q5_0 ? -16.0f : 1.0f;
};

// Orders a wave's own LDS accesses around the point where its lanes exchange data through LDS: the hardware completes
// them in program order, so all that is needed is that neither the compiler nor the instruction scheduler moves an access
// across this point (they may otherwise: the copies and the operand reads go through differently typed pointers).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int SK_APAD = 256 + 16;      // LDS row strides (+16: rows 32 apart in banks do not all collide)

__device__ __forceinline__ float f16_of(const u32x4 &v, int j) {   // j is a compile-time constant after unrolling
    const u32 u = v[j >> 1];
    return half_bits_to_float((unsigned short)((j & 1) ? (u >> 16) : (u & 0xFFFFu)));
}

// Q8_0 with nine and more activation rows, and its experts: the 256 bytes of a step go through the same 128 bytes of LDS per row, four
// blocks at a time.  With all of them in LDS a group of 16-row form takes 55 KiB, two groups per compute unit.  28672 x 8192, 16 / 32 rows
// 62.7 / 79.4 -> 62.2 / 76.6 us, 4096 x 14336, 24 rows 23.6 -> 22.4, 8 experts of 14336 x 4096, 32 slots 95.5 -> 91.4; up to eight rows the
// whole step is quicker (28672 x 8192, 8 rows 55.1 against 56.0; 32768 x 2080, 6 rows 21.3 against 23.8).
constexpr int sk_halves(int type, int ni, bool tail, bool id) { return type == MI355_Q8_0 && !tail && (ni > 1 || id) ? 2 : 1; }

// registers of one step in flight
template <int TYPE, int NI, int HALVES> struct sk_regs {
    static constexpr int NW = 32 * sk_traits<TYPE>::ROW_BYTES / 1024;   // 16-byte loads per lane for the weights
    static constexpr int NWH = NW / HALVES;                             // ... for those that are in LDS together
    static constexpr int NA = 2 * NI;                                   // ... for 8 NI activation rows of 256 bytes
    static constexpr int NT = (NI + 1) / 2;                             // ... for their 8 {d, sum} pairs each
    u32x4 w[NW], a[NA], t[NT], hdr;
    u32x4 hdr2;                             // Q4_1 / Q5_1: the second half of the eight {d, m} pairs
    u32x4 qh[2];                            // Q6_K: the high bit pairs, 32 rows x 64 bytes (on their way to LDS); Q5_0 / Q5_1: the
                                            // eight fifth-bit words of the lane's row; Q5_K ([0] only): qh bytes 16 (lane / 32) .. + 16
    u32 d6;                                 // Q6_K: the f16 super-block scale of the lane's row (hdr holds its 16 int8 scales)
    u32x4 t1;                               // Q8K: the second half of the column's block sums; its scale
    float d8;
};

// grid.x = 32-row tiles of the weight matrix, grid.y = slices of K (partial sums to `dst` as [slice][B][dst_stride] then).
// The group's four waves split the slice's steps.  TAIL: K is no multiple of 256 (per-32-block types; a form of its own, since the branch
// and its registers cost the others 7 %: Q8_0 28672 x 8192, 8 rows, 53.7 -> 57.6 us).
//
// ID: MUL_MAT_ID with a few slots per expert.  grid.y = experts, grid.z = groups that share an expert's passes (skinny_id_groups); a group
// collects its expert's (token, expert slot) pairs from the ids itself (at most SK_MAX_SLOTS of them in all: two reads of a few KiB from L2, no routing launch) and takes them 8 NI columns at a time,
// so that an expert's matrix is read from memory once however many slots chose it; the passes over further columns find their 32 rows in L2.
constexpr int SK_MAX_SLOTS = 1024;
struct sk_id {
    const int32_t *ids;        // expert of slot t * n_used + e at ids[t * ids_stride + e]
    int64_t ids_stride, expert_bytes;
    int n_used, nb1, n_slots;
};
//
// Q8K: activations in the per-super-block form of mi355_quantize_act_q8k (one scale per 256 elements, the sums of its eight 32-element
// blocks), the format ggml-cpu multiplies the super-block types with: aux1 = scales, aux2 = sums.  The integer block scales multiply the
// block sums in 24-bit integer multiply-adds and a value meets f32 once per super-block (ggml_vec_dot_q4_K_q8_K / _q5_K_ / _q6_K_ / _iq4_xs_q8_K,
// ggml/src/ggml-cpu/ggml-cpu-quants.c:6817-6848, 7539-7592, 8262-8283, 11381): 21 vector instructions per value and super-block for Q4_K
// against 32 of the Q8_1 form.
struct sk_q8k { const float *d; const _Float16 *bs; };
__device__ __forceinline__ int mul24(int a, int b) { return ((a << 8) >> 8) * ((b << 8) >> 8); }   // v_mul_i32_i24 / v_mad_i32_i24
template <int TYPE, int NI, bool TAIL, bool ID = false, bool Q8K = false>
__global__ void __launch_bounds__(256) k_mm_skinny(const uint8_t *__restrict__ W, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads,
                                                   float *__restrict__ dst, const float *__restrict__ residual, int64_t N, int K, int B,
                                                   int64_t dst_stride, int steps_per_slice, int steps_per_wave, sk_id id, sk_q8k q8) {
    typedef sk_traits<TYPE> T;
    constexpr int HALVES = sk_halves(TYPE, NI, TAIL, ID);
    typedef sk_regs<TYPE, NI, HALVES> R;
    constexpr int LDS_ROW = T::ROW_BYTES / HALVES;   // bytes of a weight row in LDS
    constexpr int WPAD = LDS_ROW + 16;
    constexpr int QHPAD = 64 + 16;
    constexpr bool Q6 = TYPE == MI355_Q6_K;
    constexpr int W_BYTES = 32 * WPAD + (Q6 ? 32 * QHPAD : 0), A_BYTES = 8 * NI * SK_APAD, T_BYTES = 8 * 8 * NI * 8;
    constexpr int G_BYTES = Q6 && !Q8K ? 16 * 8 * NI * 4 : 0;   // Q6_K: integer sums of the activation levels per 16 elements
    constexpr int WAVE_BYTES = W_BYTES + A_BYTES + T_BYTES + G_BYTES;
    constexpr int RED_BYTES = 4 * NI * 4 * 64 * 4;
    __shared__ __attribute__((aligned(16))) uint8_t s_mem[4 * WAVE_BYTES > RED_BYTES ? 4 * WAVE_BYTES : RED_BYTES];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, kh = lane >> 5;
    uint8_t *s_w = s_mem + wave * WAVE_BYTES;
    uint8_t *s_a = s_w + W_BYTES;
    float2 *s_t = (float2 *)(s_a + A_BYTES);
    int *s_g = (int *)(s_a + A_BYTES + T_BYTES);
    int *s_b = (int *)s_t;                        // Q8K: the sums of the eight blocks [8][8 NI], then the scales [8 NI] (T_BYTES hold them)
    float *s_d8 = (float *)s_t + 8 * 8 * NI;
    uint8_t *s_qh = s_w + 32 * WPAD;

    __shared__ unsigned short s_slot[ID ? SK_MAX_SLOTS : 1];
    int n_cols = B;
    int c_lo = 0;   // ID: first column of the pass
    if constexpr (ID) {
        auto expert_of = [&](unsigned sl) {
            const unsigned t = sl / (unsigned)id.n_used;
            const int ex = id.ids[t * id.ids_stride + (sl - t * (unsigned)id.n_used)];
            return ex < 0 ? 0 : (ex >= (int)gridDim.y ? (int)gridDim.y - 1 : ex);   // never index outside the expert stack
        };
        constexpr int ROUNDS = SK_MAX_SLOTS / 256;
        __shared__ int s_hits[ROUNDS][4];
        if (!Q8K || gridDim.z == 1) {   // any order: a column's sums do not depend on its neighbours
            if (threadIdx.x == 0) s_hits[0][0] = 0;
            __syncthreads();
            for (unsigned sl = threadIdx.x; sl < (unsigned)id.n_slots; sl += 256)
                if (expert_of(sl) == (int)blockIdx.y) s_slot[atomicAdd(&s_hits[0][0], 1)] = (unsigned short)sl;
            __syncthreads();
            n_cols = s_hits[0][0];
        } else {   // ascending, so that the groups that share an expert's passes agree on their columns
            uint64_t hit[ROUNDS];
#pragma unroll
            for (int i = 0; i < ROUNDS; i++) {
                const unsigned sl = (unsigned)(i * 256) + threadIdx.x;
                hit[i] = __ballot(sl < (unsigned)id.n_slots && expert_of(sl) == (int)blockIdx.y);
                if (lane == 0) s_hits[i][wave] = __popcll(hit[i]);
            }
            __syncthreads();
            int at[ROUNDS];
            n_cols = 0;
#pragma unroll
            for (int i = 0; i < ROUNDS; i++)
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    if (w == wave) at[i] = n_cols;
                    n_cols += s_hits[i][w];
                }
#pragma unroll
            for (int i = 0; i < ROUNDS; i++)
                if ((hit[i] >> lane) & 1) s_slot[at[i] + __popcll(hit[i] & ((1ull << lane) - 1))] = (unsigned short)(i * 256 + threadIdx.x);
            __syncthreads();
        }
        n_cols = __builtin_amdgcn_readfirstlane(n_cols);
        c_lo = (int)blockIdx.z * (8 * NI);
        if (n_cols <= c_lo) return;   // uniform for the whole group
        W += (int64_t)blockIdx.y * id.expert_bytes;
    }
    const int slice = ID ? 0 : (int)blockIdx.y;

    const row_layout L = make_row_layout(TYPE, K);
    const int nsteps = TAIL ? (K + 255) >> 8 : K >> 8;
    const int nblk = K >> 5;
    const int64_t row0 = (int64_t)blockIdx.x * 32;

    const int slice_lo = slice * steps_per_slice;
    const int slice_hi = slice_lo + steps_per_slice < nsteps ? slice_lo + steps_per_slice : nsteps;
    const int s_lo = slice_lo + wave * steps_per_wave;
    const int s_hi = s_lo + steps_per_wave < slice_hi ? s_lo + steps_per_wave : slice_hi;   // may be <= s_lo: a wave without steps

    // copy assignments: weights: a lane reads 16 bytes along a row, LPR lanes per row; activation rows: 16 lanes per row
    constexpr int LPR = LDS_ROW / 16, RPL = 64 / LPR;   // lanes per row, rows per load
    const int w_piece = lane % LPR, w_row = lane / LPR;
    const uint8_t *w_src[R::NWH];
#pragma unroll
    for (int u = 0; u < R::NWH; u++) {
        int64_t row = row0 + w_row + u * RPL;
        row = row < N ? row : N - 1;   // clamp: rows past the end repeat the last row and are not stored
        w_src[u] = W + row * L.row_bytes + 16 * w_piece + T::QS_OFF;
    }
    const uint8_t *qh_src[2];   // Q6_K: 4 lanes per row, 16 rows per load
#pragma unroll
    for (int u = 0; u < 2; u++) {
        int64_t row = row0 + (lane >> 2) + 16 * u;
        row = row < N ? row : N - 1;
        qh_src[u] = W + row * L.row_bytes + L.off_b + 16 * (lane & 3);
    }
    const int64_t my_row = row0 + r < N ? row0 + r : N - 1;
    const uint8_t *w_mine = W + my_row * L.row_bytes;   // the row whose results this lane holds: its scales go to registers
    auto act_row = [&](int i) -> int64_t {   // activation row of column i of the pass; columns past the end repeat the last one
        const int c = c_lo + i < n_cols ? c_lo + i : n_cols - 1;
        if constexpr (!ID) return c;
        const int sl = s_slot[c];
        return (int64_t)(sl / id.n_used) * id.nb1 + sl % id.n_used % id.nb1;
    };
    do {
    const int a_piece = lane & 15, a_row = lane >> 4;
    const int8_t *a_src[R::NA];
#pragma unroll
    for (int u = 0; u < R::NA; u++) a_src[u] = aq + act_row(a_row + 4 * u) * K + 16 * a_piece;
    const int t_piece = lane & 3, t_row = lane >> 2;   // {d, sum} pairs: 4 lanes x 16 bytes per activation row and step
    const act_ds *t_src[R::NT];
#pragma unroll
    for (int u = 0; u < R::NT; u++) t_src[u] = Q8K ? nullptr : ads + act_row(t_row + 16 * u) * nblk + 2 * t_piece;
    // Q8K: lane c < 8 NI brings the scale and the block sums of column c
    const int64_t q8_row = Q8K ? act_row(lane < 8 * NI ? lane : 0) * (K >> 8) : 0;

    // the weights of one half of a step (HALVES == 2)
    auto fetch_half = [&](int step, R &g, int half) {
        const int s = step < nsteps ? step : nsteps - 1;
#pragma unroll
        for (int u = 0; u < R::NWH; u++) g.w[half * R::NWH + u] = load16w(w_src[u] + s * T::STEP_BYTES + half * LDS_ROW);
    };
    // The last step of a row whose K is no multiple of 256: blocks past the end repeat the last one (nothing is read behind the row) and
    // get scale and minimum 0; the activation bytes they meet are those of the last block too, hence finite.
    auto fetch_tail = [&](int s, R &g) {
        constexpr int BLOCK_Q = T::ROW_BYTES / 8;   // level bytes per block
        const int last = nblk - 1;
#pragma unroll
        for (int u = 0; u < R::NWH; u++) {
            const int blk = s * 8 + 16 * w_piece / BLOCK_Q;
            g.w[u] = load16w(w_src[u] + s * T::STEP_BYTES - (blk > last ? (blk - last) * BLOCK_Q : 0));
        }
        const int so = T::FIFTH32 ? L.off_c : L.off_b;
        u32 sc[8], fw[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int blk = s * 8 + j < nblk ? s * 8 + j : last;
            if constexpr (T::PAIR) sc[j] = load4w(w_mine + so + blk * 4);
            else sc[j] = *(const unsigned short *)(w_mine + so + blk * 2);
            fw[j] = 0;
            if constexpr (T::FIFTH32) fw[j] = load4w(w_mine + L.off_b + blk * 4);
            if (s * 8 + j > last) sc[j] = 0;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            g.qh[0][j] = fw[j];
            g.qh[1][j] = fw[4 + j];
            g.hdr[j] = T::PAIR ? sc[j] : sc[2 * j] | (sc[2 * j + 1] << 16);
            g.hdr2[j] = sc[4 + j];
        }
#pragma unroll
        for (int u = 0; u < R::NA; u++) {
            const int blk = s * 8 + (a_piece >> 1);
            g.a[u] = load16(a_src[u] + s * 256 - (blk > last ? (blk - last) * 32 : 0));
        }
#pragma unroll
        for (int u = 0; u < R::NT; u++) {   // two blocks per piece; 16-byte loads of {d, sum} pairs would straddle the end of the row
            const int b0 = s * 8 + 2 * t_piece;
            const uint2 e0 = *(const uint2 *)(t_src[u] + s * 8 - (b0 > last ? b0 - last : 0)), e1 = *(const uint2 *)(t_src[u] + s * 8 + 1 - (b0 + 1 > last ? b0 + 1 - last : 0));
            g.t[u] = u32x4{e0.x, e0.y, e1.x, e1.y};
        }
    };
    // loads of one step into the register set `g` (HALVES == 2: without the weights, fetch_half)
    auto fetch = [&](int step, R &g) {
        const int s = step < nsteps ? step : nsteps - 1;
        if constexpr (TAIL) {
            if (s * 8 + 8 > nblk) {   // uniform
                fetch_tail(s, g);
                return;
            }
        }
        const int w_off = s * T::STEP_BYTES;   // < 2^31: rows are shorter than that
        if constexpr (HALVES == 1) {
#pragma unroll
            for (int u = 0; u < R::NW; u++) g.w[u] = load16w(w_src[u] + w_off);
        }
        if constexpr (T::KQ) {
            g.hdr = load16w(w_mine + w_off);
            if constexpr (TYPE == MI355_Q5_K) g.qh[0] = load16w(w_mine + w_off + 16 + 16 * kh);
        } else if constexpr (T::FIFTH32) {
            g.qh[0] = load16w(w_mine + L.off_b + s * 32);
            g.qh[1] = load16w(w_mine + L.off_b + s * 32 + 16);
            if constexpr (T::PAIR) {
                g.hdr = load16w(w_mine + L.off_c + s * 32);
                g.hdr2 = load16w(w_mine + L.off_c + s * 32 + 16);
            } else {
                g.hdr = load16w(w_mine + L.off_c + s * 16);
            }
        } else if constexpr (T::PAIR) {
            g.hdr = load16w(w_mine + L.off_b + s * 32);
            g.hdr2 = load16w(w_mine + L.off_b + s * 32 + 16);
        } else if constexpr (TYPE == MI355_IQ4_XS) {
            const u32x2 h = load8w(w_mine + L.off_b + s * 8);   // the super-block's d, scales_h, scales_l
            g.hdr[0] = h[0];
            g.hdr[1] = h[1];
        } else if constexpr (Q6) {
#pragma unroll
            for (int u = 0; u < 2; u++) g.qh[u] = load16w(qh_src[u] + s * 64);
            g.hdr = load16w(w_mine + L.off_c + s * 16);                            // sixteen int8 scales
            g.d6 = *(const unsigned short *)(w_mine + L.off_d + s * 2);
        } else {
            g.hdr = load16w(w_mine + L.off_b + s * 16);   // eight f16 block scales
        }
#pragma unroll
        for (int u = 0; u < R::NA; u++) g.a[u] = load16(a_src[u] + s * 256);
        if constexpr (Q8K) {
            g.t[0] = load16(q8.bs + (q8_row + s) * 16);
            g.t1 = load16(q8.bs + (q8_row + s) * 16 + 8);
            g.d8 = q8.d[q8_row + s];
        } else {
#pragma unroll
            for (int u = 0; u < R::NT; u++) g.t[u] = *(const u32x4_a8 *)(t_src[u] + s * 8);
        }
    };

    float acc[NI][4];
#pragma unroll
    for (int q = 0; q < NI; q++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[q][i] = 0.0f;

    // One set of load registers: as soon as a step's loads have been copied to LDS, the same registers take the next step's
    // loads, which are then in flight while this step is contracted.  Only the weight scales of the lane's row stay behind.
    R cur = {};
    if constexpr (HALVES == 2) fetch_half(s_lo, cur, 0);
    fetch(s_lo, cur);
    if constexpr (HALVES == 2) fetch_half(s_lo, cur, 1);
    for (int step = s_lo; step < s_hi; step++) {
        // ---- registers -> the wave's LDS
#pragma unroll
        for (int u = 0; u < R::NWH; u++) *(u32x4 *)(s_w + (w_row + u * RPL) * WPAD + 16 * w_piece) = cur.w[u];
        if constexpr (Q6) {
#pragma unroll
            for (int u = 0; u < 2; u++) *(u32x4 *)(s_qh + ((lane >> 2) + 16 * u) * QHPAD + 16 * (lane & 3)) = cur.qh[u];
        }
#pragma unroll
        for (int u = 0; u < R::NA; u++) {
            *(u32x4 *)(s_a + (a_row + 4 * u) * SK_APAD + 16 * a_piece) = cur.a[u];
            if constexpr (Q6 && !Q8K) {   // the lane's 16 bytes are one 16-element group of its activation row
                int sum = 0;
#pragma unroll
                for (int i = 0; i < 4; i++) sum = dot4(0x01010101, (int)cur.a[u][i], sum);
                s_g[a_piece * (8 * NI) + a_row + 4 * u] = sum;
            }
        }
        if constexpr (Q8K) {
            if (lane < 8 * NI) {
                const f16x8 lo = __builtin_bit_cast(f16x8, cur.t[0]), hi = __builtin_bit_cast(f16x8, cur.t1);   // sum = 64 hi + lo
#pragma unroll
                for (int j = 0; j < 8; j++) s_b[j * (8 * NI) + lane] = (int)(float)lo[j] + 64 * (int)(float)hi[j];
                s_d8[lane] = cur.d8;
            }
        } else {
#pragma unroll
        for (int u = 0; u < R::NT; u++) {
            if (t_row + 16 * u < 8 * NI) {
#pragma unroll
                for (int h = 0; h < 2; h++) {   // blocks 2 t_piece + h of activation row t_row + 16 u
                    const u32 d_bits = cur.t[u][2 * h], sum_bits = cur.t[u][2 * h + 1];   // copy the lanes out before bit-casting
                    const float d = __builtin_bit_cast(float, d_bits);
                    const float sum = (float)(int)sum_bits;
                    float2 v;
                    v.x = d;
                    v.y = T::OFFSET * d * sum;
                    s_t[(2 * t_piece + h) * (8 * NI) + t_row + 16 * u] = v;
                }
            }
        }
        }
        const u32x4 hdr = cur.hdr, hdr2 = cur.hdr2;
        const u32x4 fifth[2] = {cur.qh[0], cur.qh[1]};   // (Q6_K's went to LDS above)
        const u32 d6 = cur.d6;
        wave_lds_sync();
        if (step + 1 < s_hi) {
            if constexpr (HALVES == 2) fetch_half(step + 1, cur, 0);
            fetch(step + 1, cur);
        }

        const int am = r < 8 * NI ? r : r & 7;   // operand rows past the copied ones repeat copied ones; their results are not used
        if constexpr (Q8K) {
            int isum[NI][4], msum[NI][4];   // sum of scale * block sum; sum of minimum * sum of levels (Q4_K, Q5_K)
#pragma unroll
            for (int qq = 0; qq < NI; qq++)
#pragma unroll
                for (int i = 0; i < 4; i++) isum[qq][i] = msum[qq][i] = 0;
            i32x16 z;
#pragma unroll
            for (int i = 0; i < 16; i++) z[i] = 0;
            float dw, dmin = 0.0f;
            if constexpr (Q6) {
                dw = half_bits_to_float((unsigned short)d6);
#pragma unroll
                for (int hf = 0; hf < 2; hf++)
#pragma unroll
                    for (int is = 0; is < 2; is++) {
                        const u32x2 qh8 = *(const u32x2 *)(s_qh + r * QHPAD + 32 * hf + 16 * is + 8 * kh);
#pragma unroll
                        for (int qlo = 0; qlo < 2; qlo++) {
                            const u32x2 ql8 = *(const u32x2 *)(s_w + r * WPAD + 64 * hf + 32 * qlo + 16 * is + 8 * kh);
#pragma unroll
                            for (int qhi = 0; qhi < 2; qhi++) {
                                const int q = qlo + 2 * qhi, g = 8 * hf + 2 * q + is;   // as in the Q8_1 form below
                                u32x2 lv;
#pragma unroll
                                for (int i = 0; i < 2; i++) {   // level - 32 per byte: flip bit 5, then sign-extend it into bits 6 and 7
                                    const u32 t = (((ql8[i] >> (4 * qhi)) & 0x0F0F0F0Fu) | (((qh8[i] >> (2 * q)) & 0x03030303u) << 4)) ^ 0x20202020u;
                                    const u32 m = t & 0x20202020u;
                                    lv[i] = t | (m << 1) | (m << 2);
                                }
                                const u32x2 a8 = *(const u32x2 *)(s_a + am * SK_APAD + 128 * hf + 32 * q + 16 * is + 8 * kh);
                                const i32x16 D = __builtin_amdgcn_mfma_i32_32x32x16_i8(__builtin_bit_cast(long, a8), __builtin_bit_cast(long, lv), z, 0, 0, 0);
                                const u32 sc_word = hdr[g >> 2];
                                const int sc = (int)(signed char)((sc_word >> (8 * (g & 3))) & 0xFFu);
#pragma unroll
                                for (int qq = 0; qq < NI; qq++)
#pragma unroll
                                    for (int i = 0; i < 4; i++) isum[qq][i] += mul24(sc, D[4 * qq + i]);
                            }
                        }
                    }
            } else {
                int sc[8], mn[8];
                if constexpr (T::KQ) {
                    dw = half_bits_to_float((unsigned short)(hdr[0] & 0xFFFFu));
                    dmin = half_bits_to_float((unsigned short)(hdr[0] >> 16));
                    const u32 u0 = hdr[1], u1 = hdr[2], u2 = hdr[3];
                    const u32 s_lo = u0 & 0x3F3F3F3Fu, m_lo = u1 & 0x3F3F3F3Fu;
                    const u32 s_hi = (u2 & 0x0F0F0F0Fu) | (((u0 >> 6) & 0x03030303u) << 4);
                    const u32 m_hi = ((u2 >> 4) & 0x0F0F0F0Fu) | (((u1 >> 6) & 0x03030303u) << 4);
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        sc[j] = (int)(((j < 4 ? s_lo : s_hi) >> (8 * (j & 3))) & 0xFFu);
                        mn[j] = (int)(((j < 4 ? m_lo : m_hi) >> (8 * (j & 3))) & 0xFFu);
                    }
                } else {   // IQ4_XS
                    dw = half_bits_to_float((unsigned short)(hdr[0] & 0xFFFFu));
#pragma unroll
                    for (int j = 0; j < 8; j++) sc[j] = (int)(((hdr[1] >> (4 * j)) & 0xFu) | (((hdr[0] >> (16 + 2 * j)) & 3u) << 4)) - 32;
                }
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    i32x4 wop;
                    if constexpr (T::KQ) {
                        const u32x4 v = *(const u32x4 *)(s_w + r * WPAD + 32 * (j >> 1) + 16 * kh);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            wop[i] = (int)((v[i] >> (4 * (j & 1))) & 0x0F0F0F0Fu);
                            if constexpr (TYPE == MI355_Q5_K) wop[i] |= (int)(((fifth[0][i] >> j) & 0x01010101u) << 4);
                        }
                    } else {
                        const u32x4 v = *(const u32x4 *)(s_w + r * WPAD + 16 * j);
#pragma unroll
                        for (int i = 0; i < 4; i++) wop[i] = (int)iq4nl_lookup4((v[i] >> (4 * kh)) & 0x0F0F0F0Fu);
                    }
                    const i32x4 aop = *(const i32x4 *)(s_a + am * SK_APAD + 32 * j + 16 * kh);
                    const i32x16 D = __builtin_amdgcn_mfma_i32_32x32x32_i8(aop, wop, z, 0, 0, 0);
#pragma unroll
                    for (int qq = 0; qq < NI; qq++) {
                        if constexpr (T::KQ) {
                            const i32x4 b = *(const i32x4 *)(s_b + j * (8 * NI) + 8 * qq + 4 * kh);
#pragma unroll
                            for (int i = 0; i < 4; i++) msum[qq][i] += mul24(mn[j], b[i]);
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++) isum[qq][i] += mul24(sc[j], D[4 * qq + i]);
                    }
                }
            }
#pragma unroll
            for (int qq = 0; qq < NI; qq++) {
                const f32x4 d8 = *(const f32x4 *)(s_d8 + 8 * qq + 4 * kh);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float v = dw * (float)isum[qq][i];
                    if constexpr (T::KQ) v = __builtin_fmaf(-dmin, (float)msum[qq][i], v);
                    acc[qq][i] = __builtin_fmaf(d8[i], v, acc[qq][i]);
                }
            }
        } else if constexpr (Q6) {
            // 16 groups of 16 levels, each with its own int8 scale: one v_mfma_i32_32x32x16_i8 per group (8 levels per lane).
            // Group (hf, q, is): levels 128 hf + 32 q + 16 is .. + 16; level l of it = nibble q / 2 of ql byte 64 hf + 32 (q % 2) + 16 is + l
            // plus bits 2q, 2q + 1 of qh byte 32 hf + 16 is + l, minus 32 (dequantize_row_q6_K, ggml/src/ggml-quants.c:1690-1719).
            const float d = half_bits_to_float((unsigned short)d6);
#pragma unroll
            for (int hf = 0; hf < 2; hf++)
#pragma unroll
                for (int is = 0; is < 2; is++) {
                    const u32x2 qh8 = *(const u32x2 *)(s_qh + r * QHPAD + 32 * hf + 16 * is + 8 * kh);
#pragma unroll
                    for (int qlo = 0; qlo < 2; qlo++) {
                        const u32x2 ql8 = *(const u32x2 *)(s_w + r * WPAD + 64 * hf + 32 * qlo + 16 * is + 8 * kh);
#pragma unroll
                        for (int qhi = 0; qhi < 2; qhi++) {
                            const int q = qlo + 2 * qhi;
                            const int g = 8 * hf + 2 * q + is;   // scale index = position of the group in the super-block
                            u32x2 lv;
#pragma unroll
                            for (int i = 0; i < 2; i++) lv[i] = ((ql8[i] >> (4 * qhi)) & 0x0F0F0F0Fu) | (((qh8[i] >> (2 * q)) & 0x03030303u) << 4);
                            const u32x2 a8 = *(const u32x2 *)(s_a + am * SK_APAD + 128 * hf + 32 * q + 16 * is + 8 * kh);
                            i32x16 z;
#pragma unroll
                            for (int i = 0; i < 16; i++) z[i] = 0;
                            const i32x16 D = __builtin_amdgcn_mfma_i32_32x32x16_i8(__builtin_bit_cast(long, a8), __builtin_bit_cast(long, lv), z, 0, 0, 0);
                            const u32 sc_word = hdr[g >> 2];
                            const float wsg = d * (float)(int)(signed char)((sc_word >> (8 * (g & 3))) & 0xFFu);
#pragma unroll
                            for (int qq = 0; qq < NI; qq++) {
                                const float4 *e = (const float4 *)(s_t + (4 * hf + q) * (8 * NI) + 8 * qq + 4 * kh);
                                const float4 e01 = e[0], e23 = e[1];
                                const float dd[4] = {e01.x, e01.z, e23.x, e23.z};
                                const i32x4 gs = *(const i32x4 *)(s_g + g * (8 * NI) + 8 * qq + 4 * kh);
#pragma unroll
                                for (int i = 0; i < 4; i++) acc[qq][i] = __builtin_fmaf(wsg, dd[i] * (float)(D[4 * qq + i] - 32 * gs[i]), acc[qq][i]);
                            }
                        }
                    }
                }
        } else {
            // ---- per-block weight scales of this lane's row
            float ws[8], wm[8];
            if constexpr (T::KQ) {
                const float d = half_bits_to_float((unsigned short)(hdr[0] & 0xFFFFu));
                const float dmin = half_bits_to_float((unsigned short)(hdr[0] >> 16));
                    // all eight 6-bit (scale, min) pairs at once, as the bytes of four words (get_scale_min_k4, ggml-quants.c:631-638)
                const u32 u0 = hdr[1], u1 = hdr[2], u2 = hdr[3];
                const u32 s_lo = u0 & 0x3F3F3F3Fu, m_lo = u1 & 0x3F3F3F3Fu;
                const u32 s_hi = (u2 & 0x0F0F0F0Fu) | (((u0 >> 6) & 0x03030303u) << 4);
                const u32 m_hi = ((u2 >> 4) & 0x0F0F0F0Fu) | (((u1 >> 6) & 0x03030303u) << 4);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const u32 S = j < 4 ? s_lo : s_hi, M = j < 4 ? m_lo : m_hi;
                    ws[j] = d * (float)((S >> (8 * (j & 3))) & 0xFFu);
                    wm[j] = -(dmin * (float)((M >> (8 * (j & 3))) & 0xFFu));
                }
            } else if constexpr (T::PAIR) {
    #pragma unroll
                for (int j = 0; j < 8; j++) {
                    const u32 dm = j < 4 ? hdr[j & 3] : hdr2[j & 3];
                    ws[j] = half_bits_to_float((unsigned short)(dm & 0xFFFFu));
                    wm[j] = half_bits_to_float((unsigned short)(dm >> 16));
                }
            } else if constexpr (TYPE == MI355_IQ4_XS) {
    #pragma unroll
                for (int j = 0; j < 8; j++) ws[j] = iq4xs_block_scale(hdr[0], hdr[1], j);
            } else {
    #pragma unroll
                for (int j = 0; j < 8; j++) ws[j] = f16_of(hdr, j);
            }
    #pragma unroll
            for (int j = 0; j < 8; j++) {
                if constexpr (HALVES == 2) {
                    if (j == 4) {   // the second half takes the first one's place
                        // the first half's sums are formed here, not behind the branch below: sixteen registers per block less
#pragma unroll
                        for (int q = 0; q < NI; q++)
#pragma unroll
                            for (int i = 0; i < 4; i++) asm volatile("" : "+v"(acc[q][i]));
                        wave_lds_sync();
#pragma unroll
                        for (int u = 0; u < R::NWH; u++) *(u32x4 *)(s_w + (w_row + u * RPL) * WPAD + 16 * w_piece) = cur.w[R::NWH + u];
                        wave_lds_sync();
                        if (step + 1 < s_hi) fetch_half(step + 1, cur, 1);
                    }
                }
                // operand B: levels 16 kh .. + 16 of block j of weight row r
                i32x4 wop;
                if constexpr (TYPE == MI355_Q8_0) {
                    wop = *(const i32x4 *)(s_w + r * WPAD + 32 * (HALVES == 2 ? j & 3 : j) + 16 * kh);
                } else if constexpr (T::NIB32) {   // byte b of the block's 16: level b in the low nibble, level 16 + b in the high one
                    const u32x4 v = *(const u32x4 *)(s_w + r * WPAD + 16 * j);
                    const u32 fw = j < 4 ? fifth[0][j & 3] : fifth[1][j & 3];   // Q5_0 / Q5_1: bit e = fifth bit of element e
    #pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const u32 nib = (v[i] >> (4 * kh)) & 0x0F0F0F0Fu;   // elements 16 kh + 4 i .. + 4
                        if constexpr (T::TABLE) wop[i] = (int)iq4nl_lookup4(nib);
                        else if constexpr (T::FIFTH32) wop[i] = (int)(nib | spread4(fw >> (16 * kh + 4 * i)));
                        else wop[i] = (int)nib;
                    }
                } else {   // chunk j / 2: byte b of its 32: level b of sub-block 2 (j / 2) in the low nibble, of the next one in the high nibble
                    const u32x4 v = *(const u32x4 *)(s_w + r * WPAD + 32 * (j >> 1) + 16 * kh);
    #pragma unroll
                    for (int i = 0; i < 4; i++) {
                        wop[i] = (int)((v[i] >> (4 * (j & 1))) & 0x0F0F0F0Fu);
                        // Q5_K: bit j of qh byte l is the fifth bit of level l of sub-block j (dequantize_row_q5_K, ggml/src/ggml-quants.c:1482-1507)
                        if constexpr (TYPE == MI355_Q5_K) wop[i] |= (int)(((fifth[0][i] >> j) & 0x01010101u) << 4);
                    }
                }
                const i32x4 aop = *(const i32x4 *)(s_a + am * SK_APAD + 32 * j + 16 * kh);
                i32x16 z;
    #pragma unroll
                for (int i = 0; i < 16; i++) z[i] = 0;
                const i32x16 D = __builtin_amdgcn_mfma_i32_32x32x32_i8(aop, wop, z, 0, 0, 0);
    #pragma unroll
                for (int q = 0; q < NI; q++) {
                    const float4 *e = (const float4 *)(s_t + j * (8 * NI) + 8 * q + 4 * kh);
                    const float4 e01 = e[0], e23 = e[1];
                    const float dd[4] = {e01.x, e01.z, e23.x, e23.z};
                    const float xx[4] = {e01.y, e01.w, e23.y, e23.w};
    #pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float Df = (float)D[4 * q + i];
                        if constexpr (TYPE == MI355_Q4_0 || TYPE == MI355_Q5_0) {
                            acc[q][i] = __builtin_fmaf(ws[j], __builtin_fmaf(dd[i], Df, xx[i]), acc[q][i]);   // x = -8 (-16) d sum
                        } else if constexpr (TYPE == MI355_Q8_0 || T::TABLE) {
                            acc[q][i] = __builtin_fmaf(ws[j], dd[i] * Df, acc[q][i]);
                        } else {   // block minimum: + m (Q4_1, Q5_1), - dmin * 6-bit minimum (Q4_K, Q5_K)
                            acc[q][i] = __builtin_fmaf(ws[j], dd[i] * Df, acc[q][i]);
                            acc[q][i] = __builtin_fmaf(wm[j], xx[i], acc[q][i]);                              // x = d sum
                        }
                    }
                }
            }
        }
        wave_lds_sync();   // the next step's copies come after this step's reads
    }

    // the four quarters of K: fixed order 0, 1, 2, 3
    __syncthreads();   // everybody is done with the copies; the same memory now holds the partial sums
    float *s_red = (float *)s_mem;   // [wave][NI * 4][64]
#pragma unroll
    for (int q = 0; q < NI; q++)
#pragma unroll
        for (int i = 0; i < 4; i++) s_red[(wave * NI * 4 + q * 4 + i) * 64 + lane] = acc[q][i];
    __syncthreads();
    // wave w finishes the values v = w, w + 4, ...; lane (r, kh) of value (q, i) is activation row 8 q + 4 kh + i, weight row row0 + r
    for (int v = wave; v < NI * 4; v += 4) {
        const float sum = ((s_red[(0 * NI * 4 + v) * 64 + lane] + s_red[(1 * NI * 4 + v) * 64 + lane]) + s_red[(2 * NI * 4 + v) * 64 + lane]) +
                          s_red[(3 * NI * 4 + v) * 64 + lane];
        const int q = v >> 2, i = v & 3;
        const int c = c_lo + 8 * q + 4 * kh + i;
        if (c < n_cols && row0 + r < N) {
            const int64_t o = (ID ? (int64_t)s_slot[c] : (int64_t)slice * B + c) * dst_stride + row0 + r;
            dst[o] = residual ? sum + residual[o] : sum;
        }
    }
    if constexpr (ID) __syncthreads();   // the partial sums have been read: the next pass reuses the memory
    c_lo += ID ? 8 * NI * (int)gridDim.z : 8 * NI;
    } while (ID && c_lo < n_cols);
}

// sum of the K slices: dst[c][n] = sum_s part[s][c][n] (+ residual), slices in ascending order
__global__ void __launch_bounds__(256) k_skinny_slices(const float *__restrict__ part, float *__restrict__ dst, const float *__restrict__ residual,
                                                       int64_t N, int B, int64_t dst_stride, int slices) {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int c = blockIdx.y;
    if (n >= N) return;
    float sum = part[(int64_t)c * N + n];
    for (int s = 1; s < slices; s++) sum += part[((int64_t)s * B + c) * N + n];
    const int64_t o = c * dst_stride + n;
    dst[o] = residual ? sum + residual[o] : sum;
}

template <int TYPE, int NI>
void launch_skinny(hipStream_t s, const void *W, const int8_t *aq, const act_ds *ads, float *dst, const float *residual, int64_t N, int K, int B,
                   int64_t dst_stride, int slices, float *part) {
    const int nsteps = (K + 255) >> 8;
    const int steps_per_slice = (nsteps + slices - 1) / slices;
    const int steps_per_wave = (steps_per_slice + 3) / 4;
    const dim3 grid((unsigned)((N + 31) / 32), (unsigned)slices);
    float *out = slices == 1 ? dst : part;
    const float *res = slices == 1 ? residual : nullptr;
    const int64_t stride = slices == 1 ? dst_stride : N;
    constexpr bool BLOCKS32 = (sk_traits<TYPE>::NIB32 && TYPE != MI355_IQ4_XS) || TYPE == MI355_Q8_0;
    if (BLOCKS32 && K % 256 != 0)
        MI355_LAUNCH((k_mm_skinny<TYPE, NI, BLOCKS32>), grid, dim3(256), 0, s, (const uint8_t *)W, aq, ads, out, res, N, K, B, stride, steps_per_slice, steps_per_wave, sk_id{}, sk_q8k{});
    else
        MI355_LAUNCH((k_mm_skinny<TYPE, NI, false>), grid, dim3(256), 0, s, (const uint8_t *)W, aq, ads, out, res, N, K, B, stride, steps_per_slice, steps_per_wave, sk_id{}, sk_q8k{});
    if (slices > 1) {
        MI355_LAUNCH(k_skinny_slices, dim3((unsigned)((N + 255) / 256), (unsigned)B), dim3(256), 0, s, part, dst, residual, N, B, dst_stride, slices);
    }
}

template <int TYPE>
void launch_skinny_nt(hipStream_t s, const void *W, const int8_t *aq, const act_ds *ads, float *dst, const float *residual, int64_t N, int K, int B,
                      int64_t dst_stride, int slices, float *part) {
    if (B <= 8) launch_skinny<TYPE, 1>(s, W, aq, ads, dst, residual, N, K, B, dst_stride, slices, part);
    else if (B <= 16) launch_skinny<TYPE, 2>(s, W, aq, ads, dst, residual, N, K, B, dst_stride, slices, part);
    else if (B <= 24) launch_skinny<TYPE, 3>(s, W, aq, ads, dst, residual, N, K, B, dst_stride, slices, part);
    else launch_skinny<TYPE, 4>(s, W, aq, ads, dst, residual, N, K, B, dst_stride, slices, part);
}

// Groups that share an expert's passes over its columns (Q8K form; the routed tile kernels of the other types are slower than one group's
// passes).  A token chooses an expert once, so an expert has up to T columns where the average leaves it T n_used / n_expert: with one group
// per expert and row tile its passes run one after the other while the others' compute units idle.  Every token choosing the same two of 16
// experts of 2048 x 2048, 256 slots, one / two groups / routed tile kernel: Q4_K 31.0 / 25.0 / 27.0 us, Q6_K 37.2 / 28.7 / 30.0.  The second groups
// find nothing to do where the slots are spread: 25.5 -> 26.3 us there, but 48 -> 53 at 64 experts of 1024 x 2048 and 45 -> 55 at 256 of
// 512 x 2048, 1024 slots (one group, the same eight experts for every token: 33.6 and 50 us; routed 31 and 40, spread 55 and 100); up to 64 tokens
// one group is ahead of the routed kernel in either case.
int skinny_id_groups(int64_t N, int64_t n_expert, int64_t T) { return T > 64 && (N + 31) / 32 * n_expert <= 1024 ? 2 : 1; }

template <int TYPE, int NI>
void launch_skinny_id(hipStream_t s, const void *as, const int8_t *aq, const act_ds *ads, float *dst, int64_t N, int K, int64_t n_expert, const sk_id &id) {
    const int nsteps = (K + 255) >> 8;
    const dim3 grid((unsigned)((N + 31) / 32), (unsigned)n_expert);
    constexpr bool BLOCKS32 = (sk_traits<TYPE>::NIB32 && TYPE != MI355_IQ4_XS) || TYPE == MI355_Q8_0;
    if (BLOCKS32 && K % 256 != 0)
        MI355_LAUNCH((k_mm_skinny<TYPE, NI, BLOCKS32, true>), grid, dim3(256), 0, s, (const uint8_t *)as, aq, ads, dst, (const float *)nullptr, N, K, 0, N, nsteps, (nsteps + 3) / 4, id, sk_q8k{});
    else
        MI355_LAUNCH((k_mm_skinny<TYPE, NI, false, true>), grid, dim3(256), 0, s, (const uint8_t *)as, aq, ads, dst, (const float *)nullptr, N, K, 0, N, nsteps, (nsteps + 3) / 4, id, sk_q8k{});
}

template <int TYPE, int NI>
void launch_skinny_id_q8k(hipStream_t s, const void *as, const int8_t *aq, const sk_q8k &q8, float *dst, int64_t N, int K, int64_t n_expert, const sk_id &id) {
    const int nsteps = K >> 8;
    MI355_LAUNCH((k_mm_skinny<TYPE, NI, false, true, true>), dim3((unsigned)((N + 31) / 32), (unsigned)n_expert, (unsigned)skinny_id_groups(N, n_expert, id.n_slots / id.n_used)), dim3(256), 0, s, (const uint8_t *)as, aq,
                 (const act_ds *)nullptr, dst, (const float *)nullptr, N, K, 0, N, nsteps, (nsteps + 3) / 4, id, q8);
}

// slices of K: launches with fewer than ~1.5 groups per compute unit split K over several groups (and pay a second launch
// that adds the slices), as long as a slice keeps 4 steps; a short K with at most 8 activation rows is quicker in one go.
int skinny_slices(int64_t N, int64_t K, int64_t B) {
    const int64_t tiles = (N + 31) / 32, nsteps = (K + 255) >> 8;
    if (tiles >= 384 || (B <= 8 && nsteps <= 16)) return 1;
    int s = 1;
    while (s < 8 && tiles * s < 512 && nsteps / (s * 2) >= 4) s *= 2;
    return s;
}

// Columns per pass of the expert form (8, 16 or 32) by the average number of slots per expert: a few more than the average, since a second
// pass costs as much matrix work as the first, and no more than that, since every column is copied and scaled whether a slot fills it or not
constexpr int64_t SK_ID_NARROW = 5, SK_ID_WIDE = 12;

}  // namespace

}  // namespace mi355

using namespace mi355;

extern "C" {

int mi355_mul_mat_skinny_supported(int type, const void *W, int64_t K, int64_t B) {
    return is_weight_type(type) && B >= 1 && B <= 32 && K > 0 && K % type_block_elems(type) == 0 && K < (int64_t(1) << 30) && layout_loadable(W);
}

size_t mi355_mul_mat_skinny_ws_bytes(int64_t N, int64_t K, int64_t B) {
    const int s = skinny_slices(N, K, B);
    return s > 1 ? (size_t)s * B * N * sizeof(float) : 0;
}

int mi355_mul_mat_skinny(void *stream, int type, const void *W, const void *act, float *dst, const float *residual, int64_t N, int64_t K, int64_t B,
                         int64_t dst_stride, void *ws, size_t ws_bytes) {
    MI355_REQUIRE(mi355_mul_mat_skinny_supported(type, W, K, B), "mul_mat_skinny: type %d, K=%lld, B=%lld or the weight alignment is not supported", type,
                  (long long)K, (long long)B);
    MI355_REQUIRE(N > 0 && dst_stride >= N, "mul_mat_skinny: bad shape N=%lld dst_stride=%lld", (long long)N, (long long)dst_stride);
    MI355_REQUIRE(((uintptr_t)act & 15) == 0, "mul_mat_skinny: activation workspace is not 16-byte aligned");
    int slices = skinny_slices(N, K, B);
    if (slices > 1 && (ws == nullptr || ws_bytes < (size_t)slices * B * N * sizeof(float))) slices = 1;   // no room for partial sums: one slice
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + B * K);
#define X(T) launch_skinny_nt<T>(s, W, aq, ads, dst, residual, N, (int)K, (int)B, dst_stride, slices, (float *)ws);
    MI355_WEIGHT_TYPE_SWITCH(type, X)
#undef X
    return launch_status("k_mm_skinny");
}

int mi355_mul_mat_id_skinny_supported(int type, const void *as, int64_t K, int64_t n_expert, int64_t n_used, int64_t T) {
    return is_weight_type(type) && K > 0 && K % type_block_elems(type) == 0 && K < (int64_t(1) << 30) && n_expert > 0 && n_expert <= 65535 && n_used > 0 && T > 0 &&
           T * n_used <= SK_MAX_SLOTS && layout_loadable(as);
}

int mi355_mul_mat_id_skinny(void *stream, int type, const void *as, const void *act, const int32_t *ids, int64_t ids_stride, float *dst, int64_t N, int64_t K,
                            int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T) {
    MI355_REQUIRE(mi355_mul_mat_id_skinny_supported(type, as, K, n_expert, n_used, T), "mul_mat_id_skinny: type %d, K=%lld, %lld slots or the weight alignment is not supported",
                  type, (long long)K, (long long)(T * n_used));
    MI355_REQUIRE(N > 0 && nb1 > 0 && ids_stride >= n_used, "mul_mat_id_skinny: bad shape");
    MI355_REQUIRE(((uintptr_t)act & 15) == 0, "mul_mat_id_skinny: activation workspace is not 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + nb1 * T * K);
    const sk_id id = {ids, ids_stride, N * make_row_layout(type, K).row_bytes, (int)n_used, (int)nb1, (int)(T * n_used)};
    const int64_t avg = T * n_used / n_expert;   // slots per expert
#define X(TY)                                                                                 \
    if (avg <= SK_ID_NARROW) launch_skinny_id<TY, 1>(s, as, aq, ads, dst, N, (int)K, n_expert, id); \
    else if (avg <= SK_ID_WIDE) launch_skinny_id<TY, 2>(s, as, aq, ads, dst, N, (int)K, n_expert, id); \
    else launch_skinny_id<TY, 4>(s, as, aq, ads, dst, N, (int)K, n_expert, id);
    MI355_WEIGHT_TYPE_SWITCH(type, X)
#undef X
    return launch_status("k_mm_skinny (experts)");
}

int mi355_mul_mat_id_skinny_q8k(void *stream, int type, const void *as, const void *act, const int32_t *ids, int64_t ids_stride, float *dst, int64_t N,
                                int64_t K, int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T) {
    MI355_REQUIRE((type == MI355_Q4_K || type == MI355_Q5_K || type == MI355_Q6_K || type == MI355_IQ4_XS) && mi355_mul_mat_id_skinny_supported(type, as, K, n_expert, n_used, T),
                  "mul_mat_id_skinny_q8k: type %d, K=%lld, %lld slots or the weight alignment is not supported", type, (long long)K, (long long)(T * n_used));
    MI355_REQUIRE(N > 0 && nb1 > 0 && ids_stride >= n_used, "mul_mat_id_skinny_q8k: bad shape");
    MI355_REQUIRE(((uintptr_t)act & 15) == 0 && (q8k_bs_offset(K, nb1 * T) & 15) == 0, "mul_mat_id_skinny_q8k: activation workspace is not 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const sk_q8k q8 = {(const float *)(aq + q8k_d_offset(K, nb1 * T)), (const _Float16 *)(aq + q8k_bs_offset(K, nb1 * T))};
    const sk_id id = {ids, ids_stride, N * make_row_layout(type, K).row_bytes, (int)n_used, (int)nb1, (int)(T * n_used)};
    const int64_t avg = T * n_used / n_expert;   // slots per expert
#define X(TY)                                                                                           \
    if (avg <= SK_ID_NARROW) launch_skinny_id_q8k<TY, 1>(s, as, aq, q8, dst, N, (int)K, n_expert, id); \
    else if (avg <= SK_ID_WIDE) launch_skinny_id_q8k<TY, 2>(s, as, aq, q8, dst, N, (int)K, n_expert, id); \
    else launch_skinny_id_q8k<TY, 4>(s, as, aq, q8, dst, N, (int)K, n_expert, id);
    switch (type) {
        case MI355_Q4_K: X(MI355_Q4_K) break;
        case MI355_Q5_K: X(MI355_Q5_K) break;
        case MI355_IQ4_XS: X(MI355_IQ4_XS) break;
        default: X(MI355_Q6_K) break;
    }
#undef X
    return launch_status("k_mm_skinny (experts)");
}

}  // extern "C"
