// Batched quantized GEMM on the int8 matrix cores (B > 8):
//   dst[b][n] = sum_k W[n][k] * x[b][k],  W block-quantized, x quantized to Q8_1 on the device.
//
// A 256-thread group (4 waves, 2 x 2) owns a 128 (weight rows) x BN (activation rows)
// tile of dst and walks K in stages of 128 elements.  Per stage the weight rows are
// unpacked from their 4/6/8-bit blocks to int8 in LDS (each weight byte is unpacked once per
// group and reused for BN activation rows), the activation int8 rows are copied to LDS - into the
// other of two buffers, so that a stage costs one barrier - and each wave contracts its 64 x (BN/2)
// sub-tile with v_mfma_i32_32x32x32_i8, one instruction per 32-element quantization block,
// so every MFMA result is an exact per-block integer dot.  Block results are scaled by
// (weight block scale) x (activation block scale) and accumulated in f32 registers.
//
//   Q4_0 : 16 * (level - 8) as int8, scale d / 16        (one MFMA per block)
//   Q8_0 : level as int8, scale d
//   Q5_0 : level - 16 as int8, scale d;  IQ4_NL : the table value of the nibble as int8, scale d
//   IQ4_XS : as IQ4_NL, scale d * (ls - 32) from the super-block's header
//   Q4_1, Q5_1 : level 0..15 / 0..31 as int8, scale d; the "+ m * d_x * sum(q)" term of the stage's four blocks is added with two
//          v_mfma_f32_32x32x2_f32 on (dx * sum(q)) x m
//   Q4_K, Q5_K : level 0..15 / 0..31 as int8, scale d*sc; the "- dmin*m*sum(q)" term of the blocks the same way
//   Q6_K : level - 32 as int8, scale d*sc per 16 elements (two v_mfma_i32_32x32x16_i8 per block)
//
// MFMA operand mapping used here (A = activations, B = weights, D[i][j], i = activation
// row, j = weight row): lane l supplies row/column l % 32 and the k bytes
// [16*(l/32), 16*(l/32)+16) of the 32-wide step;
// D register r of lane l is element i = 8*(r/4) + 4*(l/32) + r%4, j = l % 32.  Both
// operands use the same k split, so the contraction is independent of how the hardware
// numbers k internally.
//
// Group ids are remapped so that the groups sharing one weight panel run on the same XCD
// (ids are dealt round-robin over the 8 XCDs) and hit its L2 instead of HBM.
#include "common.hpp"
#include "slices.hpp"
#include "qdot.hpp"
#include "tiles.hpp"

namespace mi355 {

constexpr int MMQ_BM = 128;          // weight rows per group
constexpr int MMQ_BK = 128;          // K elements per stage
// byte offset of 16-byte chunk c (0..7) of row r of a stage in LDS: rows of 128 bytes, the chunks of eight neighbouring rows in different
// banks (a pad of 16 bytes per row does the same, but two stages of the types with minima then leave one group per compute unit)
__device__ __forceinline__ int mmq_chunk(int r, int c) { return r * MMQ_BK + ((c ^ (r & 7)) << 4); }

// Scaling of the block sums, the larger part of the kernel's work (16 sums per lane and v_mfma_i32_32x32x32_i8, which itself takes 32 of
// the 4 x 16 x n cycles that n instructions per sum cost): the accumulator of each matrix instruction starts at the bits of
// M = 1.5 * 2^23, so that its integer result (|sum| < 2^22: 32 * 127 * 128 at most) read as a float is M + sum, without a conversion.  Then
//     t = fma(M + sum, dw, -M dw)      = sum * dw rounded once: M * dw is exact, dw has at most 19 significant bits
//     acc = fma(t, dx, acc)            dx as f16 (what block_q8_1 holds), widened inside the instruction (v_fma_mix_f32)
// two instructions per sum instead of three (convert, dw * dx, fma): see the figures at launch_mmq.  The error against 64-bit arithmetic
// stays that of three where sum * dw rarely needs more than 24 bits (Q4_0, Q5_0: 2.042e-7, 2.018e-7 of the result at K = 4096 either way; the
// types with minima gained more by their f32 form).  With levels of eight bits it would grow (Q8_0 2.027e-7 -> 2.037e-7, IQ4_NL 2.026e-7 ->
// 2.038e-7, IQ4_XS 2.030e-7 -> 2.037e-7), so for those types (mmq_cfg::WIDE) the last stage has sums of its own, which takes at least as much off
// the rounding of the long ones (it has the registers: nothing is requested any more): 1.994e-7, 1.995e-7, 1.995e-7; K = 1024, three / two
// instructions / with that: Q8_0 1.030e-7 / 1.055e-7 / 0.979e-7.  Time 114.3 -> 114.8 us (14336 x 4096, 512 rows); three instructions take 137.
constexpr float MMQ_MAGIC = 12582912.0f;
constexpr int MMQ_MAGIC_BITS = 0x4B400000;

// place of activation row r's scale in a block's row of sAd: the 16 rows of a lane (i = 8 (j / 4) + 4 (lane / 32) + j % 4 of a 32-row
// tile, j = 0..15) side by side
__device__ __forceinline__ int mmq_dx_slot(int r) { return (r & ~31) + ((r >> 2) & 1) * 16 + ((r >> 3) & 3) * 4 + (r & 3); }

template <int TYPE> struct mmq_cfg {
    static constexpr int G = TYPE == MI355_Q6_K ? 16 : 32;   // elements per weight scale
    static constexpr int NG = MMQ_BK / G;                    // weight scales per row per stage
    // a per-block offset rides on the sums of the activation levels: - dmin * m (Q4_K), + m (Q4_1, Q5_1)
    static constexpr bool MIN = TYPE == MI355_Q4_K || TYPE == MI355_Q5_K || TYPE == MI355_Q4_1 || TYPE == MI355_Q5_1;
    // 16 bytes of nibbles per block with a per-block scale: one request / commit form serves them all
    static constexpr bool NIBBLE32 = TYPE == MI355_Q4_0 || TYPE == MI355_Q4_1 || TYPE == MI355_Q5_0 || TYPE == MI355_Q5_1 || TYPE == MI355_IQ4_NL ||
                                     TYPE == MI355_IQ4_XS;
    // levels of eight bits: the last stage has sums of its own
    static constexpr bool WIDE = TYPE == MI355_Q8_0 || TYPE == MI355_IQ4_NL || TYPE == MI355_IQ4_XS;
};

// ---- a stage is requested (global -> registers) one stage ahead and committed (unpack -> LDS) while the stage before it is contracted
// sW  : int8 [MMQ_BM][MMQ_BK] (mmq_chunk)
// sWs : float [NG][MMQ_BM]   (scale g of row r at sWs[g*MMQ_BM + r])
// sWo : float [4][MMQ_BM]    (types with a block minimum: what multiplies d_x * sum(q) of the stage's 4 blocks)
// sA  : int8 [BN][MMQ_BK] (mmq_chunk);  sAd : f16 [4][BN] block scales (mmq_dx_slot);  sAs : float [4][BN]  dx*sum(q) (types with a block minimum)
// The rows a thread loads from: uniform base of the tile + a 32-bit offset per row (64-bit pointers per row are twice the registers, and
// the spills they caused took Q8_0 14336 x 4096 at 512 rows from 130 to 193 us).  A tile of 128 rows spans less than 4 GiB: launch_mmq.
__device__ __forceinline__ uint64_t uniform_addr(const void *p) {   // into scalar registers: 64-bit products of uniform values are formed by the vector ALU
    const uint64_t u = (uint64_t)p;
    return (uint64_t)(u32)__builtin_amdgcn_readfirstlane((u32)u) | ((uint64_t)(u32)__builtin_amdgcn_readfirstlane((u32)(u >> 32)) << 32);
}
template <class T> __device__ __forceinline__ T global_load(uint64_t base, u32 off) {
    return *(const T __attribute__((address_space(1))) *)(base + off);
}
template <int NR, int TPR> struct mmq_rows {
    uint64_t base;
    u32 off[NR];
    __device__ __forceinline__ void init(const uint8_t *__restrict__ W, const row_layout &L, int64_t row0, int64_t N, int tid) {
        base = uniform_addr(W + row0 * L.row_bytes);
        const int last = (int)(N - 1 - row0 < MMQ_BM - 1 ? N - 1 - row0 : MMQ_BM - 1);   // rows past the end repeat the last one and are not stored
#pragma unroll
        for (int it = 0; it < NR; it++) {
            const int r = tid / TPR + it * (256 / TPR);
            off[it] = (u32)(r < last ? r : last) * (u32)L.row_bytes;
        }
    }
};
template <int TYPE, bool NIB = mmq_cfg<TYPE>::NIBBLE32> struct mmq_wregs {};
// Q4_0, Q4_1, Q5_0, Q5_1, IQ4_NL, IQ4_XS: thread t owns blocks (row, b) = (t >> 2, t & 3) and (64 + (t >> 2), t & 3)
template <int TYPE> struct mmq_wregs<TYPE, true> : mmq_rows<2, 4> {
    static constexpr bool HAS_QH = TYPE == MI355_Q5_0 || TYPE == MI355_Q5_1;
    static constexpr bool HAS_MIN = TYPE == MI355_Q4_1 || TYPE == MI355_Q5_1;
    u32x4 q[2];
    u32 qh[2];
    u32 dm[2];   // fp16 d in the low half, fp16 m above it (HAS_MIN); IQ4_XS: the first word of the super-block's header, the second in qh
    __device__ __forceinline__ void fetch(const row_layout &L, int k0, int nblk, int tid) {
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int b = tid & 3;
            const u32 wrow = off[it];
            int blk = (k0 >> 5) + b;        // K is a multiple of 32: the last stage may hold fewer than four blocks, commit() zeroes the scales
            blk = blk < nblk ? blk : nblk - 1;
            q[it] = global_load<u32x4_a2>(base, wrow + blk * 16);
            if constexpr (HAS_QH) qh[it] = global_load<u32_a2>(base, wrow + L.off_b + blk * 4);
            const int so = HAS_QH ? L.off_c : L.off_b;   // the scales follow the fifth bits where there are any
            if constexpr (TYPE == MI355_IQ4_XS) {
                const u32x2 h = global_load<u32x2_a2>(base, wrow + L.off_b + (blk >> 3) * 8);
                dm[it] = h[0];
                qh[it] = h[1];
            } else if constexpr (HAS_MIN) dm[it] = global_load<u32_a2>(base, wrow + so + blk * 4);
            else dm[it] = global_load<unsigned short>(base, wrow + so + blk * 2);
        }
    }
    // k0: the stage that was fetched.  Nothing of a loaded value is touched before this point: a conversion at the load would wait for it.
    __device__ __forceinline__ void commit(int8_t *sW, float *sWs, float *sWo, int k0, int nblk, int tid) const {
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int r = (tid >> 2) + 64 * it, b = tid & 3;
            u32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                u32 a = q[it][i] & 0x0F0F0F0Fu, c = (q[it][i] >> 4) & 0x0F0F0F0Fu;
                if constexpr (HAS_QH) {   // bit j of qh: element j; dword i holds elements 4i.. (low nibbles) and 16 + 4i.. (high)
                    a |= spread4(qh[it] >> (4 * i));
                    c |= spread4(qh[it] >> (16 + 4 * i));
                }
                if constexpr (TYPE == MI355_Q4_0) {          // 16 * (nibble - 8): the nibble in the upper half of the byte, its top bit flipped
                    a = ((q[it][i] << 4) & 0xF0F0F0F0u) ^ 0x80808080u;
                    c = (q[it][i] & 0xF0F0F0F0u) ^ 0x80808080u;
                } else if constexpr (TYPE == MI355_Q5_0) {   // level - 16
                    a = ((a | 0x80808080u) - 0x10101010u) ^ 0x80808080u;
                    c = ((c | 0x80808080u) - 0x10101010u) ^ 0x80808080u;
                } else if constexpr (TYPE == MI355_IQ4_NL || TYPE == MI355_IQ4_XS) {
                    a = iq4nl_lookup4(a);
                    c = iq4nl_lookup4(c);
                }
                lo[i] = a;
                hi[i] = c;
            }
            *(u32x4 *)(sW + mmq_chunk(r, 2 * b)) = lo;
            *(u32x4 *)(sW + mmq_chunk(r, 2 * b + 1)) = hi;
            const u32 dm = (k0 >> 5) + b < nblk ? this->dm[it] : 0;   // past the end: scale (and minimum) 0, the block adds nothing
            if constexpr (TYPE == MI355_IQ4_XS) sWs[b * MMQ_BM + r] = iq4xs_block_scale(dm, qh[it], ((k0 >> 5) + b) & 7);
            else if constexpr (TYPE == MI355_Q4_0) sWs[b * MMQ_BM + r] = half_bits_to_float((unsigned short)(dm & 0xFFFFu)) * 0.0625f;
            else sWs[b * MMQ_BM + r] = half_bits_to_float((unsigned short)(dm & 0xFFFFu));
            if constexpr (HAS_MIN) sWo[b * MMQ_BM + r] = half_bits_to_float((unsigned short)(dm >> 16));
        }
    }
};
template <> struct mmq_wregs<MI355_Q8_0, false> : mmq_rows<4, 8> {
    u32x4 q[4];
    unsigned short d[4];
    __device__ __forceinline__ void fetch(const row_layout &L, int k0, int nblk, int tid) {
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int c = tid & 7;   // 16-byte piece of the stage
            const u32 wrow = off[it];
            int blk = (k0 >> 5) + (c >> 1);   // both pieces of a block read its scale
            blk = blk < nblk ? blk : nblk - 1;
            q[it] = global_load<u32x4_a2>(base, wrow + blk * 32 + (c & 1) * 16);
            d[it] = global_load<unsigned short>(base, wrow + L.off_b + blk * 2);
        }
    }
    __device__ __forceinline__ void commit(int8_t *sW, float *sWs, float *, int k0, int nblk, int tid) const {
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int r = (tid >> 3) + 32 * it, c = tid & 7;
            *(u32x4 *)(sW + mmq_chunk(r, c)) = q[it];
            if ((c & 1) == 0) sWs[(c >> 1) * MMQ_BM + r] = half_bits_to_float((k0 >> 5) + (c >> 1) < nblk ? d[it] : (unsigned short)0);
        }
    }
};
// Q4_K, Q5_K: stage = half a super-block, sub-blocks 4 half .. + 4, 64 B of qs per row = 4 pieces of 16 B; thread t owns the pieces
// (row, p) = (t >> 2, t & 3), (64 + (t >> 2), t & 3) and the (scale, min) of sub-block p of the stage.  Q5_K: bit j of qh[l] is the fifth bit of element l of
// sub-block j (dequantize_row_q5_K, ggml/src/ggml-quants.c:1482-1507)
template <int TYPE> struct mmq_wregs_k45 : mmq_rows<2, 4> {
    static constexpr int BB = TYPE == MI355_Q4_K ? Q4_K_BYTES : Q5_K_BYTES, QS = TYPE == MI355_Q4_K ? 16 : 48;
    u32x4 q[2], hdr[2], qh[2];
    int half;
    __device__ __forceinline__ void fetch(const row_layout &L, int k0, int, int tid) {
        half = (int)((k0 >> 7) & 1);
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int p = tid & 3;
            const u32 blk = off[it] + (k0 >> 8) * BB;
            q[it] = global_load<u32x4_a2>(base, blk + QS + (half * 2 + (p >> 1)) * 32 + (p & 1) * 16);
            hdr[it] = global_load<u32x4_a2>(base, blk);
            if constexpr (TYPE == MI355_Q5_K) qh[it] = global_load<u32x4_a2>(base, blk + 16 + (p & 1) * 16);
        }
    }
    __device__ __forceinline__ void commit(int8_t *sW, float *sWs, float *sWo, int, int, int tid) const {
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int r = (tid >> 2) + 64 * it, p = tid & 3, gl = p >> 1, h = p & 1;   // piece p: half h of group gl of the stage
            u32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                lo[i] = q[it][i] & 0x0F0F0F0Fu;
                hi[i] = (q[it][i] >> 4) & 0x0F0F0F0Fu;
                if constexpr (TYPE == MI355_Q5_K) {
                    const int ja = half * 4 + 2 * gl;   // sub-block of the low nibbles; the high nibbles are the next one
                    lo[i] |= ((qh[it][i] >> ja) & 0x01010101u) << 4;
                    hi[i] |= ((qh[it][i] >> (ja + 1)) & 0x01010101u) << 4;
                }
            }
            *(u32x4 *)(sW + mmq_chunk(r, 4 * gl + h)) = lo;
            *(u32x4 *)(sW + mmq_chunk(r, 4 * gl + 2 + h)) = hi;
            int sc, mn;
            q4k_scale_min(hdr[it][1], hdr[it][2], hdr[it][3], half * 4 + p, sc, mn);
            sWs[p * MMQ_BM + r] = half_bits_to_float((unsigned short)(hdr[it][0] & 0xFFFFu)) * (float)sc;
            sWo[p * MMQ_BM + r] = -(half_bits_to_float((unsigned short)(hdr[it][0] >> 16)) * (float)mn);
        }
    }
};
template <> struct mmq_wregs<MI355_Q4_K, false> : mmq_wregs_k45<MI355_Q4_K> {};
template <> struct mmq_wregs<MI355_Q5_K, false> : mmq_wregs_k45<MI355_Q5_K> {};
// stage = half hf of a super-block: 64 B of ql + 32 B of qh, 8 scales of 16 elements; thread t owns the 16-byte pieces (row, p) = (t >> 2, t & 3), (64 + (t >> 2), t & 3)
template <> struct mmq_wregs<MI355_Q6_K, false> : mmq_rows<2, 4> {
    u32x4 ql[2], qh[2];
    unsigned short d[2], sc[2];   // super-block scale; the int8 scales of groups 2p and 2p + 1
    __device__ __forceinline__ void fetch(const row_layout &L, int k0, int, int tid) {
        const int sb = k0 >> 8;
        const int hf = (int)((k0 >> 7) & 1);
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int p = tid & 3;
            const u32 wrow = off[it];
            ql[it] = global_load<u32x4_a2>(base, wrow + sb * 128 + hf * 64 + p * 16);
            qh[it] = global_load<u32x4_a2>(base, wrow + L.off_b + sb * 64 + hf * 32 + 16 * (p & 1));
            sc[it] = global_load<unsigned short>(base, wrow + L.off_c + sb * 16 + hf * 8 + 2 * p);
            d[it] = global_load<unsigned short>(base, wrow + L.off_d + sb * 2);
        }
    }
    __device__ __forceinline__ void commit(int8_t *sW, float *sWs, float *, int k0, int nblk, int tid) const {
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int r = (tid >> 2) + 64 * it, p = tid & 3;
            const int qa = p >> 1;
            u32x4 vA, vB;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const u32 a = (ql[it][i] & 0x0F0F0F0Fu) | (((qh[it][i] >> (2 * qa)) & 0x03030303u) << 4);
                const u32 b = ((ql[it][i] >> 4) & 0x0F0F0F0Fu) | (((qh[it][i] >> (2 * qa + 4)) & 0x03030303u) << 4);
                // level - 32 per byte: flip bit 5, then sign-extend it into bits 6..7
                const u32 ta = a ^ 0x20202020u, tb = b ^ 0x20202020u;
                const u32 ma = ta & 0x20202020u, mb = tb & 0x20202020u;
                vA[i] = ta | (ma << 1) | (ma << 2);
                vB[i] = tb | (mb << 1) | (mb << 2);
            }
            *(u32x4 *)(sW + mmq_chunk(r, 2 * qa + (p & 1))) = vA;
            *(u32x4 *)(sW + mmq_chunk(r, 2 * qa + 4 + (p & 1))) = vB;
            const float df = half_bits_to_float(d[it]);
            sWs[(2 * p) * MMQ_BM + r] = df * (float)(int)(signed char)(sc[it] & 0xFFu);
            sWs[(2 * p + 1) * MMQ_BM + r] = df * (float)(int)(signed char)(sc[it] >> 8);
        }
    }
};
template <int BN, bool WITH_SUM, bool ID> struct mmq_aregs {
    static_assert(BN == 64 || BN == 128, "columns of a tile");
    static constexpr int NQ = BN * 8 / 256, NS = BN * 4 / 256;
    uint64_t qbase, sbase;      // uniform: first row of the tile (ID: row 0)
    u32 qoff[NQ], soff[NS];     // the row as bytes / entries from there; ID: as blocks from row 0, since the gathered rows lie anywhere
    u32x4 q[NQ];
    float d[NS];
    int sum[NS];
    // row_of (ID): the activation row of every column (columns are (token, expert slot) pairs sorted by expert)
    __device__ __forceinline__ void init(const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int64_t col0, int64_t B, int nblk, int tid,
                                         const int32_t *__restrict__ row_of) {
        qbase = ID ? (uint64_t)aq : uniform_addr(aq + col0 * nblk * QK);
        sbase = ID ? (uint64_t)ads : uniform_addr(ads + col0 * nblk);
        const int last = (int)(B - 1 - col0 < BN - 1 ? B - 1 - col0 : BN - 1);   // rows past the end repeat the last one and are not stored
#pragma unroll
        for (int it = 0; it < NQ; it++) {
            const int r = (tid >> 3) + 32 * it, row = r < last ? r : last;
            qoff[it] = ID ? (u32)row_of[col0 + row] * (u32)nblk : (u32)row * (u32)(nblk * QK);
        }
#pragma unroll
        for (int it = 0; it < NS; it++) {
            const int r = (tid >> 2) + 64 * it, row = r < last ? r : last;
            soff[it] = (ID ? (u32)row_of[col0 + row] : (u32)row) * (u32)nblk;
        }
    }
    __device__ __forceinline__ void fetch(int k0, int nblk, int tid) {
        const int k = k0 + (tid & 7) * 16, k_last = nblk * QK - 16;   // past the end: any bytes, the weight scales there are 0
        const u32 kk = (u32)(k < k_last ? k : k_last);
#pragma unroll
        for (int it = 0; it < NQ; it++) q[it] = ID ? global_load<u32x4>(qbase + (uint64_t)qoff[it] * QK, kk) : global_load<u32x4>(qbase, qoff[it] + kk);
        const int blk = (k0 >> 5) + (tid & 3);
        const u32 bb = (u32)(blk < nblk ? blk : nblk - 1);
#pragma unroll
        for (int it = 0; it < NS; it++) {
            const uint64_t at = ID ? sbase + (uint64_t)(soff[it] + bb) * sizeof(act_ds) : sbase;
            const u32 o = ID ? 0 : (soff[it] + bb) * (u32)sizeof(act_ds);
            static_assert(sizeof(act_ds) == 8, "{float d; int sum;}");
            d[it] = global_load<float>(at, o);
            if constexpr (WITH_SUM) sum[it] = global_load<int>(at, o + 4);
        }
    }
    __device__ __forceinline__ void commit(int8_t *sA, _Float16 *sAd, float *sAs, int tid) const {
#pragma unroll
        for (int it = 0; it < NQ; it++) {
            const int r = (tid >> 3) + 32 * it, c = tid & 7;
            *(u32x4 *)(sA + mmq_chunk(r, c)) = q[it];
        }
#pragma unroll
        for (int it = 0; it < NS; it++) {
            const int r = (tid >> 2) + 64 * it, b = tid & 3;   // (BN is 64 or 128: every thread has a row)
            sAd[b * BN + mmq_dx_slot(r)] = (_Float16)d[it];   // exact: d is f16-rounded
            if constexpr (WITH_SUM) sAs[b * BN + r] = d[it] * (float)sum[it];
        }
    }
};

// MUL_MAT_ID with many slots (ID): column tile ct of the slot list sorted by expert (k_route_slots) holds slots [first, end) of one
// expert; their activation rows are gathered through act_row and their results go to the dst rows of dst_row.
struct mmq32_route {
    const int32_t *act_row;
    const int32_t *dst_row;
    const int32_t *tiles;      // per column tile: expert, first slot, end slot, -
    const int32_t *n_tiles;    // column tiles in use (device value)
    int64_t expert_bytes;      // from one expert's matrix to the next
};

// The matrices of a launch (up to three of one type that share the activation: Q, K and V; gate and up): their row tiles are numbered one
// matrix after the other, so that small ones fill the compute units together and pay one launch (and one sum of slices).
constexpr int MMQ_MATS = 3;
struct mmq_mat {
    const uint8_t *W;
    float *dst;
    const float *residual;     // may be null; dst's shape and stride; may be dst
    int64_t N, dst_stride;
    int first_row_tile;        // unused entries: INT_MAX
};
struct mmq_mats { mmq_mat m[MMQ_MATS]; };

typedef int i32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ long pair64(int lo, int hi) { return (long)((uint64_t)(u32)lo | (uint64_t)(u32)hi << 32); }

template <int V> struct mmq_int { static constexpr int value = V; };

// is a block scale of elements k_lo .. k_hi of the row infinite?
template <int TYPE>
__device__ __forceinline__ bool infinite_scale(const uint8_t *row, const row_layout &L, int k_lo, int k_hi) {
    constexpr bool SUPER = TYPE == MI355_Q4_K || TYPE == MI355_Q5_K || TYPE == MI355_Q6_K || TYPE == MI355_IQ4_XS;
    constexpr int EL = SUPER ? QKK : QK;
    constexpr int STRIDE = TYPE == MI355_Q4_K ? Q4_K_BYTES : TYPE == MI355_Q5_K ? Q5_K_BYTES : TYPE == MI355_IQ4_XS ? 8 : TYPE == MI355_Q4_1 || TYPE == MI355_Q5_1 ? 4 : 2;
    const uint8_t *p = row + (TYPE == MI355_Q4_K || TYPE == MI355_Q5_K ? 0 : TYPE == MI355_Q6_K ? L.off_d : TYPE == MI355_Q5_0 || TYPE == MI355_Q5_1 ? L.off_c : L.off_b);
    bool found = false;
#pragma unroll 8
    for (int b = k_lo / EL; b < (k_hi + EL - 1) / EL; b++) found |= (*(const unsigned short *)(p + (int64_t)b * STRIDE) & 0x7FFF) == 0x7C00;
    return found;
}
// the products of elements k_lo .. k_hi of a weight row and an activation row, each block sum times (weight scale * activation scale)
template <int TYPE>
__device__ __forceinline__ float plain_sum(const uint8_t *row, const row_layout &L, const int8_t *q, const act_ds *ds, int k_lo, int k_hi) {
    typedef wq<TYPE> Q;
    float sum = 0.0f;
#pragma unroll 1
    for (int c = k_lo / Q::CHUNK; c < k_hi / Q::CHUNK; c++) {
        const typename Q::chunk w = Q::load_w(row, L, c);
        const typename Q::act a = Q::load_a(q, ds, c);
        const chunk_dots i = Q::dots(w, a);
        if constexpr (TYPE == MI355_Q4_K || TYPE == MI355_Q5_K || TYPE == MI355_Q6_K) {
            sum += (float)i.i0 * ((w.d * w.scA) * a.d0) + (float)i.i1 * ((w.d * w.scB) * a.d1);
            if constexpr (TYPE != MI355_Q6_K) sum -= (w.dmin * w.mA) * a.ds0 + (w.dmin * w.mB) * a.ds1;
        } else {
            sum = Q::accumulate(sum, w, a, i);
        }
    }
    return sum;
}

template <int TYPE, int TNK, bool ID = false>
__global__ void __launch_bounds__(256, 2) k_mmq(mmq_mats mats, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int64_t K, int64_t B,
                                             row_layout L, int n_col_tiles, int n_groups, int n_groups_padded, int64_t slice_stride,
                                             mmq32_route route) {
    typedef mmq_cfg<TYPE> C;
    constexpr int BNK = 64 * TNK;
    struct stage_mem {
        __attribute__((aligned(16))) int8_t w[MMQ_BM * MMQ_BK];
        __attribute__((aligned(16))) int8_t a[BNK * MMQ_BK];
        __attribute__((aligned(16))) float ws[C::NG * MMQ_BM];
        __attribute__((aligned(16))) _Float16 ad[4 * BNK];
        __attribute__((aligned(16))) float wo[C::MIN ? MMQ_BM * 4 : 4];
        __attribute__((aligned(16))) float as[C::MIN ? BNK * 4 : 4];
    };
    __shared__ stage_mem sm[2];

    // XCD-aware id: hardware deals group ids round-robin over 8 XCDs; make logical neighbours share an XCD
    const int per_xcd = n_groups_padded >> 3;
    const int lid = ID ? (int)blockIdx.x : (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (lid >= n_groups) return;   // uniform for the whole group
    // ID: column tile by column tile over the whole chip, in the order of their work (k_route_slots), so that the last groups are the short
    // ones (8 experts of 14336 x 4096, 1024 slots: Q4_0 301 -> 238 us, Q8_0 342 -> 295; Q6_K 8 of 4096 x 2304, 600 slots 131 -> 95).  With many column
    // tiles per expert it is even: row panel by row panel on an XCD / so, 8 of 12032 x 4608, 1040 slots Q4_0 290 / 266, 4160 slots Q4_0 808 / 789, Q8_0 874 / 877;
    // 2 of 6944 x 7936, 2080 slots Q8_0 420 / 426
    // (uniform: kept in scalar registers, although the division goes through the vector ALU)
    const int per_row = ID ? n_groups / n_col_tiles : n_col_tiles;
    const int first = __builtin_amdgcn_readfirstlane(lid / per_row), second = lid - first * per_row;
    const int row_tile = ID ? second : first, col_tile = ID ? first : second;
    int mi = 0;
#pragma unroll
    for (int j = 1; j < MMQ_MATS; j++)
        if (!ID && row_tile >= mats.m[j].first_row_tile) mi = j;
    const uint8_t *W = mats.m[mi].W;
    float *dst = mats.m[mi].dst;
    const float *residual = mats.m[mi].residual;
    const int64_t N = mats.m[mi].N, dst_stride = mats.m[mi].dst_stride;
    const int64_t row0 = (int64_t)(row_tile - mats.m[mi].first_row_tile) * MMQ_BM;
    int64_t col0 = (int64_t)col_tile * BNK;
    const int32_t *row_of = nullptr;
    if constexpr (ID) {
        const int ct = col_tile;
        if (ct >= *route.n_tiles) return;   // uniform for the whole group
        W += (int64_t)route.tiles[4 * ct] * route.expert_bytes;
        col0 = route.tiles[4 * ct + 1];
        B = route.tiles[4 * ct + 2];
        row_of = route.act_row;
    }

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, lhi = lane >> 5;
    const int wrow0 = (wave & 1) * 64;           // weight rows of this wave inside the tile

    // split K: grid row y walks stages [k_lo, k_hi) and writes its sums to slice y of `dst` (a workspace then, see launch_mmq)
    const int nblk = (int)(K >> 5), stages = (nblk + MMQ_BK / QK - 1) / (MMQ_BK / QK), st_per = (stages + (int)gridDim.y - 1) / (int)gridDim.y;
    const int s_lo = (int)blockIdx.y * st_per, s_hi = s_lo + st_per < stages ? s_lo + st_per : stages;
    if (gridDim.y > 1) dst += (int64_t)blockIdx.y * slice_stride;

    // ID: a tile whose columns all lie in its first half (the second tile of an expert that is routed a few more than 128 slots) runs with
    // half the columns per wave: half the matrix instructions and sums to scale (8 experts of 14336 x 4096: Q8_0, 1400 slots 463 -> 377 us,
    // Q4_0, 1024 slots 342 -> 330).  Uniform for the whole group.  Not for batches: their groups mostly run in one round, whose time is
    // that of the full tiles (Q4_0 14336 x 4096, 160 rows: 63 us with and without, 512 rows 99.5 -> 100.2 for the larger kernel).
    auto walk = [&](auto tn) __attribute__((always_inline)) {
        constexpr int TN = decltype(tn)::value, BN = 64 * TN;
        const int wcol0 = (wave >> 1) * (32 * TN);   // activation rows of this wave inside the tile
        f32x16 acc[TN][2];
    #pragma unroll
        for (int tb = 0; tb < TN; tb++)
    #pragma unroll
            for (int tw = 0; tw < 2; tw++)
    #pragma unroll
                for (int r = 0; r < 16; r++) acc[tb][tw][r] = 0.0f;

        i32x16 magic;
    #pragma unroll
        for (int r = 0; r < 16; r++) magic[r] = MMQ_MAGIC_BITS;

        mmq_wregs<TYPE> wregs;
        mmq_aregs<BN, C::MIN, ID> aregs;
        wregs.init(W, L, row0, N, threadIdx.x);
        aregs.init(aq, ads, col0, B, nblk, threadIdx.x, row_of);
        auto fetch = [&](int st) {
            wregs.fetch(L, st * MMQ_BK, nblk, threadIdx.x);
            aregs.fetch(st * MMQ_BK, nblk, threadIdx.x);
        };
        auto commit = [&](stage_mem &m, int st) {
            wregs.commit(m.w, m.ws, m.wo, st * MMQ_BK, nblk, threadIdx.x);
            aregs.commit(m.a, m.ad, m.as, threadIdx.x);
        };

        // operands and scales of one Q8_1 block for the wave's tiles
        constexpr int NS = C::G == 32 ? 1 : 2;   // scale groups per block
        struct block_ops { i32x4 a[TN], w[2]; };
        struct block_scales {
            f16x8 dx[TN][2];     // activation block scales of this lane's 16 rows per tile
            float dw[2][NS];
        };
        int a_at = NS == 1 ? mmq_chunk(wcol0 + l32, lhi) : mmq_chunk(wcol0 + l32, 0) + 8 * lhi;
        int w_at = NS == 1 ? mmq_chunk(wrow0 + l32, lhi) : mmq_chunk(wrow0 + l32, 0) + 8 * lhi;
        // one 16-byte chunk per lane half (2 ks + lhi); two groups of 16 (Q6_K): this lane half's 8 bytes of both groups' chunks
        auto load_op = [&](const int8_t *m, int at, int ks) {
            if constexpr (NS == 1) return *(const i32x4 *)(m + (at ^ (ks << 5)));
            else {
                const i32x2 g0 = *(const i32x2 *)(m + (at ^ (ks << 5))), g1 = *(const i32x2 *)(m + (at ^ (ks << 5) ^ 16));
                return i32x4{g0[0], g0[1], g1[0], g1[1]};
            }
        };
        auto load_ops = [&](const stage_mem &m, int ks) {
            block_ops f;
    #pragma unroll
            for (int tb = 0; tb < TN; tb++) f.a[tb] = load_op(m.a + tb * 32 * MMQ_BK, a_at, ks);
    #pragma unroll
            for (int tw = 0; tw < 2; tw++) f.w[tw] = load_op(m.w + tw * 32 * MMQ_BK, w_at, ks);
            return f;
        };
        auto load_scales = [&](const stage_mem &m, int ks) {
            block_scales f;
    #pragma unroll
            for (int tb = 0; tb < TN; tb++)
    #pragma unroll
                for (int h = 0; h < 2; h++) f.dx[tb][h] = *(const f16x8 *)(m.ad + ks * BN + wcol0 + tb * 32 + 16 * lhi + 8 * h);
    #pragma unroll
            for (int tw = 0; tw < 2; tw++)
    #pragma unroll
                for (int h = 0; h < NS; h++) f.dw[tw][h] = m.ws[(ks * NS + h) * MMQ_BM + wrow0 + tw * 32 + l32];
            return f;
        };
        // matrix instruction n of a block: tile (tb, tw), scale group h.  Two groups of 16 (Q6_K): one v_mfma_i32_32x32x16_i8 each (the
        // 32-element form with half of the weights zeroed costs the vector ALU four more instructions).
        constexpr int NM = TN * 2 * NS;
        auto mma = [&](const block_ops &f, int n) {
            const int tb = n / NS % TN, tw = n / NS / TN, h = n % NS;
            if constexpr (NS == 1) return __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a[tb], f.w[tw], magic, 0, 0, 0);
            else return __builtin_amdgcn_mfma_i32_32x32x16_i8(pair64(f.a[tb][2 * h], f.a[tb][2 * h + 1]), pair64(f.w[tw][2 * h], f.w[tw][2 * h + 1]), magic, 0, 0, 0);
        };
        auto scale = [&](const block_scales &f, int n, const i32x16 &I) {
            const int tb = n / NS % TN, tw = n / NS / TN, h = n % NS;
            const float dw = f.dw[tw][h], mdw = -MMQ_MAGIC * dw;
    #pragma unroll
            for (int r = 0; r < 16; r++) {
                const int bits = I[r];
                acc[tb][tw][r] = __builtin_fmaf(__builtin_fmaf(__builtin_bit_cast(float, bits), dw, mdw), (float)f.dx[tb][r >> 3][r & 7], acc[tb][tw][r]);
            }
        };

        fetch(s_lo);
        commit(sm[0], s_lo);
        fetch(s_lo + 1 < s_hi ? s_lo + 1 : s_lo);
        __syncthreads();
        int buf = 0, st = s_lo;
        f32x16 before[C::WIDE ? TN : 1][2];   // WIDE: the sums of all but the last stage
        const bool two = C::WIDE && (nblk & 3) == 1 && s_hi == stages && s_hi - s_lo > 1;   // ... the last two, where the last holds one block
    #pragma unroll
        for (int part = 0; part < (C::WIDE ? 2 : 1); part++) {
            const int part_end = C::WIDE && part == 0 ? s_hi - 1 - two : s_hi;
            if constexpr (C::WIDE) {
                if (part == 1) {
    #pragma unroll
                    for (int tb = 0; tb < TN; tb++)
    #pragma unroll
                        for (int tw = 0; tw < 2; tw++)
    #pragma unroll
                            for (int r = 0; r < 16; r++) {
                                before[tb][tw][r] = acc[tb][tw][r];
                                acc[tb][tw][r] = 0.0f;
                            }
                    if (two) {   // (both buffers before the sums: the requested stage's registers make room for them)
                        commit(sm[buf ^ 1], s_hi - 1);
                        __syncthreads();
                    }
                }
            }
            for (; st < part_end; st++, buf ^= 1) {
                const stage_mem &m = sm[buf];
                asm volatile("" : "+v"(a_at), "+v"(w_at));   // the four chunk addresses of a stage are formed in the loop: kept across it they cost spills
                // One matrix instruction is always in flight: its successor is issued before its sums are scaled, so that neither waits for the
                // other (left to the compiler, all of them write the same registers one after the other); the next block's operands are read
                // from LDS while the last sums of this one are scaled.
                block_ops f = load_ops(m, 0);
                block_scales sc = load_scales(m, 0);
                i32x16 I = mma(f, 0);
    #pragma unroll
                for (int ks = 0; ks < 4; ks++) {
                    block_scales sc_next = sc;
    #pragma unroll
                    for (int n = 0; n < NM; n++) {
                        const i32x16 cur = I;
                        I = mma(f, n + 1 < NM ? n + 1 : 0);   // (the last one of a stage is not used)
                        __builtin_amdgcn_sched_barrier(0);
                        if (n == NM - 2 && ks < 3) f = load_ops(m, ks + 1);
                        if (n == NM - 1 && ks < 3) sc_next = load_scales(m, ks + 1);
                        scale(sc, n, cur);
                        asm volatile("" : "+v"(acc[n / NS % TN][n / NS / TN]));   // formed here, and not behind the matrix instructions of the whole stage
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    sc = sc_next;
                }
                if constexpr (C::MIN) {
                    // acc += sum_b (dx * sum q)[i][b] * m[j][b] over the 4 blocks of the stage (Q4_K, Q5_K: m = -dmin * 6-bit minimum): two
                    // v_mfma_f32_32x32x2_f32 per tile on the matrix pipe, which waits for the vector ALUs anyway; k = lane / 32.  In f32 as the
                    // batch-1 kernels do it (as f16 operands the term carried 3.6e-4 of the result).
    #pragma unroll
                    for (int p = 0; p < 2; p++) {
                        float af[TN], bf[2];
    #pragma unroll
                        for (int tb = 0; tb < TN; tb++) af[tb] = m.as[(2 * p + lhi) * BN + wcol0 + tb * 32 + l32];
    #pragma unroll
                        for (int tw = 0; tw < 2; tw++) bf[tw] = m.wo[(2 * p + lhi) * MMQ_BM + wrow0 + tw * 32 + l32];
    #pragma unroll
                        for (int tb = 0; tb < TN; tb++)
    #pragma unroll
                            for (int tw = 0; tw < 2; tw++) acc[tb][tw] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[tb], bf[tw], acc[tb][tw], 0, 0, 0);
                    }
                }
                if (part == 0 && st + 1 < s_hi) {   // the next stage, requested one stage ago, goes to the other buffer (uniform)
                    commit(sm[buf ^ 1], st + 1);
                    fetch(st + 2 < s_hi ? st + 2 : st + 1);   // past the end the last stage is requested again and never used
                    __syncthreads();
                }
            }
        }
        if constexpr (C::WIDE) {
    #pragma unroll
            for (int tb = 0; tb < TN; tb++)
    #pragma unroll
                for (int tw = 0; tw < 2; tw++)
    #pragma unroll
                    for (int r = 0; r < 16; r++) acc[tb][tw][r] += before[tb][tw][r];
        }

        // An infinite weight scale makes a sum M * inf - M * inf: where a wave's sums are not all finite, the NaNs of rows with such a scale are
        // formed again, block by block (a NaN of another origin stays one).  Four chains; the test takes up to 1 % of a call, at each store 2 to 4.
        float zero[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    #pragma unroll
        for (int tb = 0; tb < TN; tb++)
    #pragma unroll
            for (int tw = 0; tw < 2; tw++)
    #pragma unroll
                for (int r = 0; r < 16; r++) zero[r & 3] = __builtin_fmaf(acc[tb][tw][r], 0.0f, zero[r & 3]);
        if (__ballot((zero[0] + zero[1]) + (zero[2] + zero[3]) != 0.0f) != 0) {   // uniform
            const int k_lo = s_lo * MMQ_BK, k_hi = s_hi * MMQ_BK < K ? s_hi * MMQ_BK : (int)K;
            bool infinite[2];
    #pragma unroll
            for (int tw = 0; tw < 2; tw++) {
                const int64_t n = row0 + wrow0 + tw * 32 + l32;
                infinite[tw] = n < N && infinite_scale<TYPE>(W + n * L.row_bytes, L, k_lo, k_hi);
            }
            if (__ballot(infinite[0] || infinite[1]) != 0) {   // uniform
    #pragma unroll 1
                for (int i = 0; i < TN * 32; i++) {   // sum r of tile (tb, tw)
                    const int r = i & 15, tw = (i >> 4) & 1;
                    const int64_t n = row0 + wrow0 + tw * 32 + l32, b = col0 + wcol0 + (i >> 5) * 32 + 8 * (r >> 2) + 4 * lhi + (r & 3);
                    if (!(tw ? infinite[1] : infinite[0]) || b >= B) continue;
                    const int64_t arow = ID ? (int64_t)row_of[b] : b;
                    const float sum = plain_sum<TYPE>(W + n * L.row_bytes, L, aq + arow * K, ads + arow * nblk, k_lo, k_hi);
    #pragma unroll
                    for (int j = 0; j < TN * 32; j++) {
                        const float at = acc[j >> 5][(j >> 4) & 1][j & 15];
                        acc[j >> 5][(j >> 4) & 1][j & 15] = j == i && at != at ? sum : at;
                    }
                }
            }
        }
        // store: lane holds weight row j = l32 of each 32-wide tile, 16 activation rows
    #pragma unroll
        for (int tb = 0; tb < TN; tb++)
    #pragma unroll
            for (int tw = 0; tw < 2; tw++) {
                const int64_t n = row0 + wrow0 + tw * 32 + l32;
    #pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int64_t b = col0 + wcol0 + tb * 32 + 8 * (r >> 2) + 4 * lhi + (r & 3);
                    if (n < N && b < B) {
                        const int64_t o = (ID ? (int64_t)route.dst_row[b] : b) * dst_stride + n;
                        dst[o] = residual ? acc[tb][tw][r] + residual[o] : acc[tb][tw][r];
                    }
                }
            }
    };
    if constexpr (ID) {
        if (B - col0 <= BNK / 2) {
            walk(mmq_int<1>{});
            return;
        }
    }
    walk(mmq_int<TNK>{});
}

// What bounds the kernel is the vector ALU: a wave issues 637 of its instructions per stage, 512 of them the two per block sum and 16
// matrix instructions, which are busy a quarter of that time (counters, Q4_0 14336 x 4096, 512 rows; 4 cycles each = 2550 cycles of the
// 2800 a stage takes with one group per compute unit).  Before the two-instruction form, the double-buffered stages and the f32 minima, by
// type (14336 x 4096, 512 rows with the quantization launch, us): Q4_0 124 -> 98, Q4_1 228 -> 128, Q5_0 149 -> 124, Q5_1 229 -> 140,
// IQ4_NL 149 -> 128, Q8_0 146 -> 130; 64 rows: Q4_0 34.3 -> 32.3.  Q6_K with 16-element instead of masked 32-element matrix
// instructions: 4096 x 11008, 64 rows 41.2 -> 39.5.
//
static size_t mmq_slab_bytes(int n, int64_t rows, int64_t B) { return (size_t)n * (size_t)rows * (size_t)B * sizeof(float); }

// A product with few tiles leaves most of the chip idle while each group walks all of K: such launches are cut along K into
// slices that run side by side and a second launch adds the slices in fixed order.  At least four stages per slice, at most
// eight slices, at most two groups per compute unit; more of them, up to sixteen, where a model of the time in us says so, which a sweep of n = 1 .. 16 over
// (1024 .. 21603 rows, 10 .. 112 stages, 50 .. 512 columns) meets within some 15 %: a stage takes 1.2 (64 columns) or 2.1 (128), Q6_K 1.7 times that; 1.4
// times with a second group on the compute unit; the sum 4, and 8 bytes per value and slice at 4 TB/s.  A call, us: Q6_K 1135 x 7424, 65 rows
// 41.2 -> 30.9 (16 slices instead of 8), Q5_1 3509 x 1216, 73 rows 23.6 -> 18.9 (5 instead of 2).  Groups are counted as an XCD gets them, padded to eighths: 18
// tiles in 12 slices are 36 on the 32 units of one (Q4_0 1115 x 11776, 184 rows 42.0 us; in 8 slices 39.5).  From 600 tiles on, where the whole chip is busy
// twice over, the model's steps no longer tell (Q4_0 28743 x 6400, 326 rows 231 us uncut, 264 in two; Q4_1 20630 x 5888, 481 rows 251 and 284; on the
// other side of the line Q4_1 18629 x 7168, 415 rows 301 and 276).  A short last slice of the fewest does not count: Q4_1 5309 x 3392, 231 rows in six slices (five
// stages each, two in the last) 42.7 us, in seven 48.3; Q8_0 4755 x 2176, 144 rows in four 29.4, in six 32.4.  Up to two thirds of the others are short where the second
// round is of padding only: Q4_0 2477 x 4096, 626 rows, 100 tiles in five slices (seven stages, four in the last) 49.1, in eight 53.4; with 20 of 22 stages in the last
// Q5_1 2537 x 13792, 527 rows in five 149, in nine 124.  (Fewer slices than these would be quicker here
// and there, Q5_0 8491 x 2016, 316 rows 49.9 -> 44.5 with one instead of two, but make longer f32 sums.)
// ws_bytes: what is there for the partial sums; none of them fits: one slice.
static int mmq_slices(int type, int64_t row_tiles, int64_t K, int64_t B, int64_t rows, size_t ws_bytes) {
    const int64_t bn = B <= 64 ? 64 : 128;
    const int64_t groups = row_tiles * ((B + bn - 1) / bn), stages = (K + MMQ_BK - 1) / MMQ_BK;
    int64_t least = 512 / groups;
    if (least > stages / 4) least = stages / 4;
    if (least > 8) least = 8;
    if (least < 1) least = 1;
    least = (stages + (stages + least - 1) / least - 1) / ((stages + least - 1) / least);   // no empty slice
    const float stage = (bn == 64 ? 1.2f : 2.1f) * (type == MI355_Q6_K ? 1.7f : 1.0f);
    int64_t best = 1;
    float best_us = 0.0f;
    const int64_t most = groups < 600 ? 16 : least;
    for (int64_t n = least; n <= most && n <= stages; n++) {
        const int64_t per = (stages + n - 1) / n, g = (groups + 7) / 8 * 8 * n;
        if (n > 1 && mmq_slab_bytes((int)n, rows, B) > ws_bytes) break;
        if ((stages + per - 1) / per != n) continue;
        // the fewest slices, whose last one is short: its groups run beside or behind the others and do not count
        const int64_t last = stages - (n - 1) * per;
        const bool is_short = 2 * last <= per || (3 * last <= 2 * per && groups * n <= 512 && g > 512);
        const int64_t at_once = n == least && n > 1 && is_short ? g / n * (n - 1) : g;
        const float busy = at_once <= 256 ? 1.0f : 1.4f * (float)((at_once + 511) / 512);
        const float us = (float)per * stage * busy + (n > 1 ? 4.0f + (float)(n * rows * B) * 8.0f / 4e6f : 0.0f);
        if (n == least || us < 0.95f * best_us) {
            best = n;
            best_us = us;
        }
    }
    return (int)best;
}
static int64_t mmq_row_tiles(int n_mats, const int64_t *Ns) {
    int64_t t = 0;
    for (int i = 0; i < n_mats; i++) t += (Ns[i] + MMQ_BM - 1) / MMQ_BM;
    return t;
}
static size_t mmq_ws_bytes(int n_mats, const int64_t *Ns, int64_t K, int64_t B) {   // for any type
    int64_t rows = 0;
    for (int i = 0; i < n_mats; i++) rows += Ns[i];
    const int64_t row_tiles = mmq_row_tiles(n_mats, Ns);
    const int a = mmq_slices(MI355_Q4_0, row_tiles, K, B, rows, SIZE_MAX), b = mmq_slices(MI355_Q6_K, row_tiles, K, B, rows, SIZE_MAX), n = a > b ? a : b;
    return n > 1 ? mmq_slab_bytes(n, rows, B) : 0;
}

// dst[b][n] of every matrix = sum of its slices in ascending order (+ residual).  part: [slice][B][rows of all matrices]; one activation row per blockIdx.y (rows beyond its range in turn)
constexpr int64_t MMQ_SUM_ROWS = 65535;
__device__ __forceinline__ const mmq_mat &mmq_mat_of(const mmq_mats &mats, int64_t &n) {
    int j = 0;
    while (j < MMQ_MATS - 1 && n >= mats.m[j].N) n -= mats.m[j++].N;
    return mats.m[j];
}
__global__ void __launch_bounds__(256) k_mmq_split_sum(const float *__restrict__ part, mmq_mats mats, int64_t rows, int64_t B, int n_slices) {
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= rows) return;
    int64_t n = r;
    const mmq_mat &m = mmq_mat_of(mats, n);
    for (int64_t b = blockIdx.y; b < B; b += MMQ_SUM_ROWS) {
        float acc = part[b * rows + r];
        for (int sl = 1; sl < n_slices; sl++) acc = add_rn(acc, part[((int64_t)sl * B + b) * rows + r]);
        const int64_t o = b * m.dst_stride + n;
        m.dst[o] = m.residual ? add_rn(acc, m.residual[o]) : acc;
    }
}
// ... four neighbouring elements per lane, for matrices of N % 4 == 0 with 16-byte aligned rows in dst and residual (4096 x 333, five slices: 9.3 -> 6.6 us)
template <int SL>
__global__ void __launch_bounds__(256) k_mmq_split_sum4(const float *__restrict__ part, mmq_mats mats, int64_t rows, int64_t B, int n_slices) {
    const int64_t r = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (r >= rows) return;
    int64_t n = r;
    const mmq_mat &m = mmq_mat_of(mats, n);
    for (int64_t b = blockIdx.y; b < B; b += MMQ_SUM_ROWS) {
        slab_sum<SL> slabs;
        slabs.request(part + b * rows + r, rows * B, n_slices);
        const int64_t o = b * m.dst_stride + n;
        f32x4 acc = slabs.sum(part + b * rows + r, rows * B, n_slices);
        if (m.residual) {
            const f32x4 t = *(const f32x4 *)(m.residual + o);
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] = add_rn(acc[j], t[j]);
        }
        *(f32x4 *)(m.dst + o) = acc;
    }
}
static void launch_mmq_split_sum(hipStream_t s, const float *part, const mmq_mats &mats, int n_mats, int64_t rows, int64_t B, int n_slices) {
    bool wide = true;
    for (int i = 0; i < n_mats; i++) {
        const mmq_mat &m = mats.m[i];
        wide = wide && m.N % 4 == 0 && m.dst_stride % 4 == 0 && (((uintptr_t)m.dst | (uintptr_t)m.residual) & 15) == 0;
    }
    wide = wide && (rows + 1023) / 1024 * B >= 256;   // a group per compute unit at least: 1024 rows, 64 activation rows, 16 slabs, the whole product 16.1 us by one, 16.6 by four elements per lane
    const int64_t per = wide ? 1024 : 256;
    const dim3 grid((unsigned)((rows + per - 1) / per), (unsigned)(B < MMQ_SUM_ROWS ? B : MMQ_SUM_ROWS));
    if (!wide) {
        MI355_LAUNCH(k_mmq_split_sum, grid, dim3(256), 0, s, part, mats, rows, B, n_slices);
        return;
    }
#define MI355_SUM_LAUNCH(SL) MI355_LAUNCH(k_mmq_split_sum4<SL>, grid, dim3(256), 0, s, part, mats, rows, B, n_slices)
    MI355_SLAB_SWITCH(n_slices, MI355_SUM_LAUNCH)
#undef MI355_SUM_LAUNCH
}

// The kernel reaches the 128 rows of a tile by 32-bit offsets from its first one: K up to some 2^25.  Longer rows run on the byte-load kernels.
static bool mmq_rows_fit(int type, int64_t K) {
    const int64_t row = make_row_layout(type, K).row_bytes;
    return MMQ_BM * (row > K ? row : K) <= (int64_t(1) << 32);
}

template <int TYPE, int TN>
static void launch_mmq(hipStream_t s, int n_mats, const mi355_gemv_mat *mats, const void *act, int64_t K, int64_t B, void *ws, size_t ws_bytes) {
    constexpr int BN = 64 * TN;
    const row_layout L = make_row_layout(TYPE, K);
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + B * K);
    mmq_mats a, part;
    int64_t Ns[MMQ_MATS], rows = 0;
    int row_tiles = 0;
    for (int i = 0; i < MMQ_MATS; i++) {
        if (i >= n_mats) {
            a.m[i] = mmq_mat{nullptr, nullptr, nullptr, 0, 0, 0x7fffffff};
            part.m[i] = a.m[i];
            continue;
        }
        const mi355_gemv_mat &m = mats[i];
        a.m[i] = mmq_mat{(const uint8_t *)m.W, m.dst, m.residual, m.N, m.dst_stride, row_tiles};
        part.m[i] = mmq_mat{(const uint8_t *)m.W, (float *)ws + rows, nullptr, m.N, 0, row_tiles};
        Ns[i] = m.N;
        rows += m.N;
        row_tiles += (int)((m.N + MMQ_BM - 1) / MMQ_BM);
    }
    for (int i = 0; i < n_mats; i++) part.m[i].dst_stride = rows;
    const int n_col_tiles = (int)((B + BN - 1) / BN);
    const int n_groups = row_tiles * n_col_tiles;
    const int n_groups_padded = (n_groups + 7) & ~7;
    const int n_slices = mmq_slices(TYPE, row_tiles, K, B, rows, ws == nullptr || ((uintptr_t)ws & 15) != 0 ? 0 : ws_bytes);
    const dim3 grid((unsigned)n_groups_padded, (unsigned)n_slices);
    MI355_LAUNCH((k_mmq<TYPE, TN>), grid, dim3(256), 0, s, n_slices > 1 ? part : a, aq, ads, K, B, L, n_col_tiles, n_groups, n_groups_padded, rows * B, mmq32_route{});
    if (n_slices > 1) launch_mmq_split_sum(s, (const float *)ws, a, n_mats, rows, B, n_slices);
}

template <int TYPE>
static void launch_mmq_tn(hipStream_t s, int n_mats, const mi355_gemv_mat *mats, const void *act, int64_t K, int64_t B, void *ws, size_t ws_bytes) {
    if (B <= 64) launch_mmq<TYPE, 1>(s, n_mats, mats, act, K, B, ws, ws_bytes);
    else launch_mmq<TYPE, 2>(s, n_mats, mats, act, K, B, ws, ws_bytes);
}

// the routed launch: 128-column tiles over the slot list sorted by expert; the routing workspace is laid out as for the
// super-block kernel's routed form (act_row[S], dst_row[S], tiles[4 x ((S + 63) / 64 + n_expert)], n_tiles)
template <int TYPE>
static void launch_mmq_id(hipStream_t s, const void *as, const int8_t *aq, const act_ds *ads, const int32_t *ids, int64_t ids_stride, float *dst, int64_t N, int64_t K,
                          int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T, void *route_ws) {
    constexpr int BN = 128;
    const int64_t S = T * n_used;
    const int max_tiles = (int)((S + BN - 1) / BN + n_expert);
    int32_t *act_row = (int32_t *)route_ws, *dst_row = act_row + S, *tiles = dst_row + S, *n_tiles = tiles + 4 * ((S + 63) / 64 + n_expert);
    launch_route_slots(s, ids, ids_stride, n_expert, n_used, nb1, T, BN, act_row, dst_row, tiles, n_tiles);
    const row_layout L = make_row_layout(TYPE, K);
    const int n_row_tiles = (int)((N + MMQ_BM - 1) / MMQ_BM);
    const int n_groups = n_row_tiles * max_tiles;
    const int n_groups_padded = (n_groups + 7) & ~7;
    const mmq32_route route = {act_row, dst_row, tiles, n_tiles, N * L.row_bytes};
    mmq_mats a;
    for (int i = 0; i < MMQ_MATS; i++) a.m[i] = i ? mmq_mat{nullptr, nullptr, nullptr, 0, 0, 0x7fffffff} : mmq_mat{(const uint8_t *)as, dst, nullptr, N, N, 0};
    MI355_LAUNCH((k_mmq<TYPE, 2, true>), dim3((unsigned)n_groups_padded), dim3(256), 0, s, a, aq, ads, K, S, L, max_tiles, n_groups, n_groups_padded, (int64_t)0, route);
}

}  // namespace mi355

using namespace mi355;

extern "C" int mi355_mul_mat_id_q_supported(int type, const void *as, int64_t N, int64_t K, int64_t n_expert) {
    const bool typed = type == MI355_Q4_0 || type == MI355_Q4_1 || type == MI355_Q5_0 || type == MI355_Q5_1 || type == MI355_IQ4_NL ||
                       type == MI355_Q8_0 || type == MI355_Q6_K || type == MI355_IQ4_XS;
    if (!typed || N <= 0 || K <= 0 || K >= (int64_t(1) << 30) || K % type_block_elems(type) != 0 || n_expert <= 0 || n_expert > 256) return 0;
    return layout_loadable(as) ? 1 : 0;
}

extern "C" int mi355_mul_mat_id_q(void *stream, int type, const void *as, const void *act, const int32_t *ids, int64_t ids_stride, float *dst, int64_t N,
                                  int64_t K, int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T, void *route_ws, size_t route_ws_bytes) {
    MI355_REQUIRE(mi355_mul_mat_id_q_supported(type, as, N, K, n_expert), "mul_mat_id_q: type %d, K=%lld, %lld experts or the weight alignment is not supported",
                  type, (long long)K, (long long)n_expert);
    MI355_REQUIRE(n_used > 0 && nb1 > 0 && T > 0 && ids_stride >= n_used, "mul_mat_id_q: bad shape");
    MI355_REQUIRE(T * n_used < (1 << 24) && nb1 * T < (1 << 24), "mul_mat_id_q: too many slots");
    MI355_REQUIRE(((uintptr_t)act & 15) == 0, "mul_mat_id_q: activation workspace is not 16-byte aligned");
    if (!mmq_rows_fit(type, K)) return mi355_mul_mat_id_vec(stream, type, as, act, ids, ids_stride, dst, N, K, n_expert, n_used, nb1, T);
    const size_t need = mi355_mul_mat_id_q8k_route_bytes(n_expert, n_used, T);
    if (route_ws == nullptr || route_ws_bytes < need || ((uintptr_t)route_ws & 15) != 0) {
        set_error("mul_mat_id_q: routing workspace of %zu bytes, need %zu (16-byte aligned)", route_ws_bytes, need);
        return MI355_ERR_WORKSPACE;
    }
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + nb1 * T * K);
    // the kernel counts the activation's blocks in 32 bits: tokens in runs of fewer than 2^32 of them (one run up to 137 GB of activations)
    const int64_t run = ((int64_t(1) << 32) - 1) / (nb1 * (K / QK));
    MI355_REQUIRE(run > 0, "mul_mat_id_q: nb1=%lld rows per token are too many", (long long)nb1);
    for (int64_t t0 = 0; t0 < T; t0 += run) {
        const int64_t n = T - t0 < run ? T - t0 : run;
#define X(TY) \
    case TY: launch_mmq_id<TY>(s, as, aq + t0 * nb1 * K, ads + t0 * nb1 * (K / QK), ids + t0 * ids_stride, ids_stride, dst + t0 * n_used * N, N, K, n_expert, n_used, nb1, n, route_ws); break;
        switch (type) { X(MI355_Q4_0) X(MI355_Q4_1) X(MI355_Q5_0) X(MI355_Q5_1) X(MI355_Q6_K) X(MI355_IQ4_XS) X(MI355_IQ4_NL) X(MI355_Q8_0) }
#undef X
    }
    return launch_status("k_mmq (routed)");
}

extern "C" size_t mi355_mul_mat_q_multi_ws_bytes(int n_mats, const int64_t *Ns, int64_t K, int64_t B) {
    if (n_mats < 1 || n_mats > MMQ_MATS || K <= 0 || B <= 0 || K % QK != 0) return 0;
    for (int i = 0; i < n_mats; i++)
        if (Ns[i] <= 0) return 0;
    return mmq_ws_bytes(n_mats, Ns, K, B);
}
extern "C" size_t mi355_mul_mat_q_ws_bytes(int64_t N, int64_t K, int64_t B) { return mi355_mul_mat_q_multi_ws_bytes(1, &N, K, B); }

extern "C" int mi355_mul_mat_q(void *stream, int type, const void *W, const void *act, float *dst, int64_t N, int64_t K,
                               int64_t B, int64_t dst_stride) {
    return mi355_mul_mat_q_ws(stream, type, W, act, dst, N, K, B, dst_stride, nullptr, 0);
}

extern "C" int mi355_mul_mat_q_ws(void *stream, int type, const void *W, const void *act, float *dst, int64_t N, int64_t K,
                                  int64_t B, int64_t dst_stride, void *ws, size_t ws_bytes) {
    const mi355_gemv_mat m = {type, W, N, dst, dst_stride, nullptr};
    return mi355_mul_mat_q_multi(stream, type, 1, &m, act, K, B, ws, ws_bytes);
}

extern "C" int mi355_mul_mat_q_multi(void *stream, int type, int n_mats, const mi355_gemv_mat *mats, const void *act, int64_t K, int64_t B, void *ws,
                                     size_t ws_bytes) {
    MI355_REQUIRE(is_weight_type(type), "mul_mat_q: unsupported weight type %d", type);
    MI355_REQUIRE(n_mats >= 1 && n_mats <= MMQ_MATS, "mul_mat_q: 1..%d matrices per launch, got %d", MMQ_MATS, n_mats);
    MI355_REQUIRE(K > 0 && B > 0, "mul_mat_q: bad shape K=%lld B=%lld", (long long)K, (long long)B);
    MI355_REQUIRE(K % type_block_elems(type) == 0, "mul_mat_q: K=%lld is not a multiple of the block size", (long long)K);
    int64_t row_tiles = 0;
    bool fit = mmq_rows_fit(type, K);
    for (int i = 0; i < n_mats; i++) {
        MI355_REQUIRE(mats[i].type == type, "mul_mat_q: the matrices of a launch have one type");
        MI355_REQUIRE(mats[i].N > 0, "mul_mat_q: bad shape N=%lld", (long long)mats[i].N);
        MI355_REQUIRE(mats[i].dst_stride >= mats[i].N, "mul_mat_q: dst_stride < N");
        row_tiles += (mats[i].N + MMQ_BM - 1) / MMQ_BM;
        fit = fit && layout_loadable(mats[i].W);
    }
    if (!fit) {   // a matrix at an odd address, rows beyond 32-bit offsets
        for (int i = 0; i < n_mats; i++) {
            const int rc = gemv_unaligned((hipStream_t)stream, type, mats[i].W, act, mats[i].dst, mats[i].residual, mats[i].N, K, B, mats[i].dst_stride);
            if (rc != MI355_OK) return rc;
        }
        return MI355_OK;
    }
    MI355_REQUIRE(((uintptr_t)act & 15) == 0, "mul_mat_q: activation workspace is not 16-byte aligned");
    MI355_REQUIRE(row_tiles * ((B + 63) / 64) < (1 << 30), "mul_mat_q: too many tiles");
    hipStream_t s = (hipStream_t)stream;
#define MI355_MMQ_LAUNCH(TY) launch_mmq_tn<TY>(s, n_mats, mats, act, K, B, ws, ws_bytes);
    MI355_WEIGHT_TYPE_SWITCH(type, MI355_MMQ_LAUNCH)
#undef MI355_MMQ_LAUNCH
    return launch_status("k_mmq");
}
