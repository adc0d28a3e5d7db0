// FLASH_ATTN_EXT for one query token over a long KV cache (head size 128, up to four query heads per kv head): the streaming
// form, for f16 caches (k_fattn_dec_stream, described here) and for Q8_0 / Q4_0 caches in the device row layout
// (k_fattn_dec_stream_q, further down).
//
// The kernel is bound by how many bytes of K and V a compute unit keeps in flight, not by arithmetic: a token reads every cell
// once and does 4 flops per byte.  So a wave owns a contiguous range of 64-cell tiles of one kv head and moves them with
// global-to-LDS transfers (no registers in between) into its own two-stage ring: while tile t is worked on, tile t + 1 (32 KiB:
// 64 K rows, 64 V rows) is on its way and tile t + 2 is requested as soon as t's last LDS read has returned.  Two waves share a
// compute unit (2 x 2 x 32 KiB of LDS), 512 waves the chip; no barrier anywhere, every wave writes its own partial result
// (running maximum, sum, un-normalised output) and k_fattn_combine merges them.
//
// Per tile a lane stands for one cell.  Scores: v_mfma_f32_4x4x4f16 works on sixteen independent 4 x 4 blocks, block b = lanes
// 4b .. 4b + 3; lane l supplies row l % 4 of A and column l % 4 of B and receives column l % 4 of D with the rows in its four
// registers.  With A = q (row = query head, the same in every block) and B = K^T (column = cell 4b + l % 4 = l) the four scores
// of cell l land in lane l's registers after 32 steps over the head dimension: no padding columns, no cross-lane sums.  The
// soft-max update is then ordinary per-lane arithmetic on 64 cells at once with one wave-wide maximum per head.  Output:
// the same instruction with A = P (row = head, k = four consecutive cells, read back from a 512-byte transposed copy in LDS)
// and B = V (k = cell, column = element l or 64 + l), whose operand - four cells at one element - is a transposing LDS read
// (ds_read_b64_tr_b16) of the row-major V tile.
//
// LDS layout of a stage: K rows at row * 256 with 16-byte chunk c of row r stored at chunk position c ^ (r & 15), so that the
// 64 lanes reading chunk c of their own rows hit all banks; V rows row-major.  Both are written by transfers that cover four
// whole rows each (fully coalesced in HBM); the permutation happens in the choice of the global address per lane.
#include "common.hpp"
#include "fattn.hpp"

#include <float.h>

namespace mi355 {

constexpr int FS_TILE = 64;                    // cells per tile
constexpr int FS_D = 128;                      // head size
constexpr int FS_ROW = FS_D * 2;               // bytes of a K or V row
constexpr int FS_KT = FS_TILE * FS_ROW;        // bytes of a K (or V) tile
constexpr int FS_STAGE = 2 * FS_KT;
constexpr int FS_WAVES = 2;                    // per group (= per compute unit)
constexpr int FS_MAX_TILES = 64;               // tiles per wave: its mask values are fetched into LDS up front
constexpr int FS_TOTAL_WAVES = 512;

#define FS_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (7 << 4) | (0xF << 8))

// Running soft-max state of a wave: per lane the sums of its own cells' weights; the maxima and the outputs are wave-wide.
struct fs_state {
    float m[4], lsum[4];
    f32x4 o0, o1;   // elements lane and 64 + lane of heads 0..3
};
__device__ __forceinline__ void fs_init(fs_state &S) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
        S.m[r] = -FLT_MAX / 2;
        S.lsum[r] = 0.0f;
    }
    S.o0 = f32x4{0.f, 0.f, 0.f, 0.f};
    S.o1 = f32x4{0.f, 0.f, 0.f, 0.f};
}
// q of the group's four heads, 512 values, eight per lane (head lane / 16, elements 8 (lane % 16) .. + 7; zeros past the R heads): requested ahead of the transfers,
// because a wave's loads return in the order of their issue.  (Every lane loading all 128 values of head lane % 4 behind the first tiles came to a third of a wave's
// instructions over one tile, and none of them could run before those tiles had landed.)
__device__ __forceinline__ void fs_request_q(const uint8_t *__restrict__ q, size_t q_nb2, int64_t head0, int R, int lane, f32x4 (&x)[2]) {
    const int h = lane >> 4;
    const float *qp = (const float *)(q + (head0 + (h < R ? h : 0)) * q_nb2) + (lane & 15) * 8;
    x[0] = *(const f32x4 *)qp;
    x[1] = *(const f32x4 *)(qp + 4);
}
// ... as f16 pairs, rounded as the reference rounds q to the K type (ggml-cpu.c:11037-11040), through FS_QLDS bytes of the wave's LDS: qv = the 128 values of head
// lane % 4.  Inline assembly, as all LDS accesses beside transfers in flight; heads FS_QROW bytes apart, so that the four of them lie in different banks.
constexpr int FS_QROW = FS_ROW + 16, FS_QLDS = 4 * FS_QROW;
__device__ __forceinline__ void fs_spread_q(f32x4 (&x)[2], int R, int lane, unsigned q_lds, u32 (&qv)[FS_D / 2]) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const f16x2 p = {(_Float16)x[i >> 1][2 * (i & 1)], (_Float16)x[i >> 1][2 * (i & 1) + 1]};
        w[i] = (lane >> 4) < R ? __builtin_bit_cast(u32, p) : 0u;
    }
    asm volatile("ds_write_b128 %0, %1" ::"v"(q_lds + (unsigned)(lane >> 4) * FS_QROW + (unsigned)(lane & 15) * 16u), "v"(w) : "memory");
    u32x4 t[16];
#pragma unroll
    for (int i = 0; i < 16; i++) asm volatile("ds_read_b128 %0, %1" : "=v"(t[i]) : "v"(q_lds + (unsigned)(lane & 3) * FS_QROW + (unsigned)i * 16u));
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]), "+v"(t[4]), "+v"(t[5]), "+v"(t[6]), "+v"(t[7]), "+v"(t[8]), "+v"(t[9]), "+v"(t[10]), "+v"(t[11]),
                   "+v"(t[12]), "+v"(t[13]), "+v"(t[14]), "+v"(t[15]));
#pragma unroll
    for (int i = 0; i < 16; i++) {
        qv[4 * i] = t[i][0];
        qv[4 * i + 1] = t[i][1];
        qv[4 * i + 2] = t[i][2];
        qv[4 * i + 3] = t[i][3];
    }
}
// The mask values of a wave's cells, eight per lane and step (cells past the end count as masked): requested ahead of the transfers, then into the wave's LDS at m_lds
template <int MT>   // tiles the wave has room for
__device__ __forceinline__ void fs_request_mask(const fattn_args &a, int64_t c_begin, int n, int lane, u32x4 (&mc)[MT / 8]) {
    const unsigned short *mrow = (const unsigned short *)a.mask;
    const bool wide = ((uintptr_t)mrow & 15) == 0;
#pragma unroll
    for (int it = 0; it < MT / 8; it++) {
        const int j = it * 64 + lane;
        const int64_t c = c_begin + (int64_t)j * 8;
        mc[it] = u32x4{0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u};   // -inf
        if (j * 8 < n * FS_TILE) {
            if (mrow && wide && c + 8 <= a.Nkv) {
                mc[it] = load16(mrow + c);
            } else {
                unsigned short e[8];
#pragma unroll
                for (int i = 0; i < 8; i++) e[i] = c + i < a.Nkv ? (mrow ? mrow[c + i] : (unsigned short)0) : (unsigned short)0xFC00;
#pragma unroll
                for (int i = 0; i < 4; i++) mc[it][i] = (u32)e[2 * i] | ((u32)e[2 * i + 1] << 16);
            }
        }
    }
}
template <int MT>
__device__ __forceinline__ void fs_store_mask(u32x4 (&mc)[MT / 8], int lane, unsigned m_lds) {
#pragma unroll
    for (int it = 0; it < MT / 8; it++) asm volatile("ds_write_b128 %0, %1" ::"v"(m_lds + (unsigned)(it * 64 + lane) * 16u), "v"(mc[it]) : "memory");
}
// ALiBi slopes of the four heads (ggml-cpu.c:10998-11003), wave-uniform
__device__ __forceinline__ void fs_slopes(const fattn_args &a, int64_t head0, float (&slope)[4]) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
        slope[r] = 1.0f;
        if (a.max_bias > 0.0f) {
            const unsigned h = (unsigned)(head0 + r);
            slope[r] = h < a.n_head_log2 ? powf(a.m0, (float)(h + 1)) : powf(a.m1, (float)(2 * (h - a.n_head_log2) + 1));
        }
    }
}
// The soft-max update of the state with one tile's raw scores (q . k of this lane's cell and the four heads), and P^T (head, cell)
// as f16 into the wave's 512 bytes of LDS at p_wr (= base + 2 * lane), where fs_output reads it back as the A operand.  LDS serves a
// wave's operations in order: those reads see these writes, and the next tile's writes come after them.
// P32: as f32, 256 bytes per head, for fs_output_f32
template <int NH = 4, bool P32 = false>   // NH: heads the group has at most
__device__ __forceinline__ void fs_softmax(const float (&raw)[4], float mv, float scale, float softcap, const float (&slope)[4], unsigned p_wr, fs_state &S) {
    constexpr float NEG = -FLT_MAX / 2;
    const bool valid = mv != -INFINITY;
#pragma unroll
    for (int r = 0; r < NH; r++) {
        float sc = raw[r] * scale;
        if (softcap != 0.0f) sc = softcap * tanhf(sc);
        sc += slope[r] * mv;
        sc = valid ? sc : NEG;
        const float mn = fmaxf(S.m[r], wave_max_dpp(sc));
        const float f = __expf(S.m[r] - mn);
        S.m[r] = mn;
        const float p = valid ? __expf(sc - mn) : 0.0f;
        S.lsum[r] = S.lsum[r] * f + p;
        S.o0[r] *= f;
        S.o1[r] *= f;
        if constexpr (P32) {
            *(float __attribute__((address_space(3))) *)(uintptr_t)(p_wr + (unsigned)(r * FS_TILE * 4)) = p;
        } else {
            const u32 ph = float_to_half_bits(p);
            asm volatile("ds_write_b16 %0, %1 offset:%2" ::"v"(p_wr), "v"(ph), "n"(r * FS_TILE * 2) : "memory");
        }
    }
}
// Scores of one tile (kc: the 16 chunks of this lane's K row), then fs_softmax.
template <int NH = 4, bool P32 = false>
__device__ __forceinline__ void fs_scores(const u32 (&qv)[FS_D / 2], const u32x4 (&kc)[16], float mv, float scale, float softcap, const float (&slope)[4],
                                          unsigned p_wr, fs_state &S) {
    constexpr int CH = P32 ? 8 : 2;   // chains of matrix operations, added as a tree
    f32x4 sc[CH];
#pragma unroll
    for (int i = 0; i < CH; i++) sc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 16; c++) {
        const u32 a0 = qv[4 * c], a1 = qv[4 * c + 1], a2 = qv[4 * c + 2], a3 = qv[4 * c + 3];
        const u32 b0 = kc[c][0], b1 = kc[c][1], b2 = kc[c][2], b3 = kc[c][3];
        const u32x2 qa = {a0, a1}, qb = {a2, a3}, ka = {b0, b1}, kb2 = {b2, b3};
        f32x4 &s0 = sc[2 * c % CH], &s1 = sc[(2 * c + 1) % CH];
        s0 = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, qa), __builtin_bit_cast(f16x4, ka), s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, qb), __builtin_bit_cast(f16x4, kb2), s1, 0, 0, 0);
    }
    float raw[4];
#pragma unroll
    for (int r = 0; r < 4; r++) raw[r] = CH == 2 ? sc[0][r] + sc[1][r] : ((sc[0][r] + sc[1 % CH][r]) + (sc[2 % CH][r] + sc[3 % CH][r])) + ((sc[4 % CH][r] + sc[5 % CH][r]) + (sc[6 % CH][r] + sc[7 % CH][r]));
    fs_softmax<NH, P32>(raw, mv, scale, softcap, slope, p_wr, S);
}
// This lane's offset inside a row-major V tile for the transposing reads of fs_output: lane l' = lane % 16 of its 16-lane group
// g points at row c0 + l' / 4, elements 16 g + 4 (l' % 4) .. + 3
__device__ __forceinline__ unsigned fs_v_lane(int lane) {
    return (unsigned)((lane & 15) >> 2) * FS_ROW + (unsigned)((lane >> 4) * 16 + (lane & 3) * 4) * 2;
}
// Output of one tile: four cells per step, elements lane and 64 + lane; every operand of the tile is requested before the first
// is used.  v_addr: LDS byte address of the V tile + fs_v_lane; p_rd: the wave's P^T + 128 * (lane % 4).
template <int NJ = 16>   // steps of four cells: 16 = a whole tile, 8 = half of one
__device__ __forceinline__ void fs_output(unsigned v_addr, unsigned p_rd, fs_state &S) {
    u32x2 vlo[NJ], vhi[NJ], pa[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const unsigned addr = v_addr + (unsigned)(j * 4 * FS_ROW);
        asm volatile("ds_read_b64 %0, %1" : "=v"(pa[j]) : "v"(p_rd + (unsigned)(j * 8)));
        asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(vlo[j]) : "v"(addr));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:128" : "=v"(vhi[j]) : "v"(addr));
    }
#pragma unroll
    for (int jb = 0; jb < NJ; jb += 8)   // the wait names its registers so that nothing is used ahead of it; 24 operands per statement
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(vlo[jb]), "+v"(vlo[jb + 1]), "+v"(vlo[jb + 2]), "+v"(vlo[jb + 3]), "+v"(vlo[jb + 4]), "+v"(vlo[jb + 5]), "+v"(vlo[jb + 6]), "+v"(vlo[jb + 7]),
                       "+v"(vhi[jb]), "+v"(vhi[jb + 1]), "+v"(vhi[jb + 2]), "+v"(vhi[jb + 3]), "+v"(vhi[jb + 4]), "+v"(vhi[jb + 5]), "+v"(vhi[jb + 6]), "+v"(vhi[jb + 7]),
                       "+v"(pa[jb]), "+v"(pa[jb + 1]), "+v"(pa[jb + 2]), "+v"(pa[jb + 3]), "+v"(pa[jb + 4]), "+v"(pa[jb + 5]), "+v"(pa[jb + 6]), "+v"(pa[jb + 7]));
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        S.o0 = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, pa[j]), __builtin_bit_cast(f16x4, vlo[j]), S.o0, 0, 0, 0);
        S.o1 = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, pa[j]), __builtin_bit_cast(f16x4, vhi[j]), S.o1, 0, 0, 0);
    }
}

// The same for one half of the elements (H = 0: lane, 1: 64 + lane), same sums
template <int H> __device__ __forceinline__ void fs_output_half(unsigned v_addr, unsigned p_rd, f32x4 &o) {
    constexpr int NJ = 16;
    u32x2 v[NJ], pa[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const unsigned addr = v_addr + (unsigned)(j * 4 * FS_ROW);
        asm volatile("ds_read_b64 %0, %1" : "=v"(pa[j]) : "v"(p_rd + (unsigned)(j * 8)));
        if constexpr (H == 0) asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(v[j]) : "v"(addr));
        else asm volatile("ds_read_b64_tr_b16 %0, %1 offset:128" : "=v"(v[j]) : "v"(addr));
    }
#pragma unroll
    for (int jb = 0; jb < NJ; jb += 8)
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(v[jb]), "+v"(v[jb + 1]), "+v"(v[jb + 2]), "+v"(v[jb + 3]), "+v"(v[jb + 4]), "+v"(v[jb + 5]), "+v"(v[jb + 6]), "+v"(v[jb + 7]),
                       "+v"(pa[jb]), "+v"(pa[jb + 1]), "+v"(pa[jb + 2]), "+v"(pa[jb + 3]), "+v"(pa[jb + 4]), "+v"(pa[jb + 5]), "+v"(pa[jb + 6]), "+v"(pa[jb + 7]));
#pragma unroll
    for (int j = 0; j < NJ; j++) o = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, pa[j]), __builtin_bit_cast(f16x4, v[j]), o, 0, 0, 0);
}
// One half of the elements (v_lane: that half of the row-major V tile + fs_v_lane) with the probabilities as f32: o[r] = sum over the tile's cells of p[r][cell] * V[cell] at the
// lane's element, each product and sum rounded once, as the vector kernel does it.  V comes from the transposing reads, four cells each; p is NH x 64 floats.  Four chains of sixteen
// cells, added as a tree.  One head: 64 multiply-adds that take V as f16, p read by all lanes at one address.  More: the matrix instruction for f32 (lane = row lane % 4 of P and column
// lane % 4 of V, as in fs_output, one cell per step), which serves four heads at once.  Four heads with
// multiply-adds: 512 / 128 heads, 256 cells 8.0 us, with the matrix instruction 7.5.
template <int NH> __device__ __forceinline__ void fs_output_f32(const uint8_t __attribute__((address_space(3))) *v_lane, const float __attribute__((address_space(3))) *p, int lane, f32x4 &o) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const float __attribute__((address_space(3))) *mine = p + (NH > 1 && (lane & 3) < NH ? lane & 3 : 0) * FS_TILE;   // rows past the group's heads repeat the first one and are not used
    float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FS_TILE / 4; j++) {
        const f16x4 v = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(v_lane + j * 4 * FS_ROW)));
        const f32x4 pr = *(const f32x4 __attribute__((address_space(3))) *)(mine + 4 * j);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (NH == 1) sum[i] = __builtin_fmaf(pr[i], (float)v[i], sum[i]);
            else acc[i] = __builtin_amdgcn_mfma_f32_4x4x1f32(pr[i], (float)v[i], acc[i], 0, 0, 0);
        }
    }
    if constexpr (NH == 1) {
        o[0] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    } else {
#pragma unroll
        for (int r = 0; r < NH; r++) o[r] = (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
    }
}

// The states of a group's waves (at most NWV) meet in LDS: one partial result per group.  all: `stride` floats per wave, whose LDS reads lie behind it; head r's
// result goes to out + r * head_step.
template <int NWV>
__device__ __forceinline__ void fs_join(const fs_state &S, float *all, int stride, float *out, int64_t head_step, int R, int lane, int wave) {
    asm volatile("" ::: "memory");   // the reads of fs_output come first
    float *mine = all + wave * stride;   // [4][FS_D], maxima, sums
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float L = wave_sum_dpp(S.lsum[r]);
        mine[r * FS_D + lane] = S.o0[r];
        mine[r * FS_D + 64 + lane] = S.o1[r];
        if (lane == 0) {
            mine[4 * FS_D + r] = S.m[r];
            mine[4 * FS_D + 4 + r] = L;
        }
    }
    __syncthreads();
    const int n_waves = (int)(blockDim.x >> 6);
    for (int idx = wave; idx < 2 * R; idx += n_waves) {   // half a head per wave and turn
        const int r = idx >> 1, d = 64 * (idx & 1) + lane;
        float m[NWV], l[NWV], o[NWV];   // all requested before any is used; past the last wave its values again, left out below
#pragma unroll
        for (int w = 0; w < NWV; w++) {
            const float *part = all + (w < n_waves ? w : n_waves - 1) * stride;
            m[w] = part[4 * FS_D + r];
            l[w] = part[4 * FS_D + 4 + r];
            o[w] = part[r * FS_D + d];
        }
        float M = m[0], L = 0.0f, O = 0.0f;
#pragma unroll
        for (int w = 1; w < NWV; w++) M = fmaxf(M, m[w]);
#pragma unroll
        for (int w = 0; w < NWV; w++) {
            if (w >= n_waves) break;   // uniform
            const float f = __expf(m[w] - M);
            L += l[w] * f;
            O += o[w] * f;
        }
        float *p = out + r * head_step;
        p[d] = O;
        if (d == 0) {
            p[FS_D] = M;
            p[FS_D + 1] = L;
        }
    }
}

// ONE: no wave has more than one tile; it keeps one stage, three or four waves fit where two walked two tiles each, and they join their states (us a call:
// 32 / 8 heads, 5120 cells 14.5 -> 13.3, 6144 15.2 -> 14.2, 8192 16.2 -> 15.8; 16 / 4 heads, 12288 16.2 -> 14.6, 16384 17.6 -> 16.3; 4 / 4 heads, 16384 15.9 -> 13.5)
constexpr int FS_WAVES_ONE = 4;
template <bool ONE>
__global__ void __launch_bounds__((ONE ? FS_WAVES_ONE : FS_WAVES) * 64, 1) k_fattn_dec_stream(fattn_args a, int tiles_per_wave, int n_tiles, int R) {
    constexpr int NWV = ONE ? FS_WAVES_ONE : FS_WAVES, STAGES = ONE ? 1 : 2, MT = ONE ? 8 : FS_MAX_TILES;
    __shared__ __attribute__((aligned(1024))) uint8_t ring_buf[NWV * STAGES * FS_STAGE];
    __shared__ __attribute__((aligned(16))) unsigned short pbuf[NWV][4][FS_TILE];
    __shared__ __attribute__((aligned(16))) unsigned short mbuf[NWV][MT * FS_TILE];
    __shared__ __attribute__((aligned(16))) uint8_t qbuf[NWV][FS_QLDS];
    // the ring is written by global-to-LDS transfers only
    asm volatile("" ::"v"((void *)ring_buf) : "memory");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int split = (int)blockIdx.x * (ONE ? (int)(blockDim.x >> 6) : FS_WAVES) + wave;   // ONE: the launch may give a group fewer than four waves
    const int64_t hk = blockIdx.y;
    const int t_begin = split * tiles_per_wave;
    const int t_end = t_begin + tiles_per_wave < n_tiles ? t_begin + tiles_per_wave : n_tiles;
    const int n = t_end > t_begin ? t_end - t_begin : 0;
    const int64_t c_begin = (int64_t)t_begin * FS_TILE;

    float slope[4];
    fs_slopes(a, hk * R, slope);
    uint8_t *ring = ring_buf + wave * (STAGES * FS_STAGE);
    // transfers of tile t into stage st: instruction i moves rows 4i .. 4i + 3; lane p -> row 4i + p / 16, chunk position p % 16.
    // A whole tile in range: scalar row addresses plus per-lane offsets that are the same for every tile; the last, partial tile
    // of the cache clamps its rows per lane (rows past the end repeat the last cell; their scores are discarded).
    const int rsub = lane >> 4, pos = lane & 15;
    unsigned koff[4], voff;
#pragma unroll
    for (int vv = 0; vv < 4; vv++) koff[vv] = (unsigned)rsub * (unsigned)a.k_nb1 + (unsigned)((pos ^ ((4 * vv + rsub) & 15)) << 4);
    voff = (unsigned)rsub * (unsigned)a.v_nb1 + (unsigned)(pos << 4);
    const uint8_t *k_head = a.k + hk * a.k_nb2, *v_head = a.v + hk * a.v_nb2;
    auto dma = [&](const uint8_t *g, unsigned off, uint8_t *l) {   // g, l: wave-uniform
        buf_to_lds16(g, off, 0, l);
    };
    // which = 0: the K half of the stage, 1: the V half (sixteen transfers each).  The cell they start at; rows past the end of the cache repeat the last cell
    auto issue_clamped = [&](int64_t c0, int st, int which) {
        uint8_t *hb = ring + st * FS_STAGE + which * FS_KT;
        const int64_t nb1 = which ? (int64_t)a.v_nb1 : (int64_t)a.k_nb1;
        const uint8_t *g = (which ? v_head : k_head) + c0 * nb1;
        const int last = a.Nkv - c0 < FS_TILE ? (int)(a.Nkv - 1 - c0) : FS_TILE - 1;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int row = 4 * i + rsub;
            dma(g, (unsigned)(row < last ? row : last) * (unsigned)nb1 + (unsigned)((which ? pos : (pos ^ (row & 15))) << 4), hb + i * 1024);
        }
    };
    auto issue = [&](int t, int st, int which) {
        const int64_t c0 = c_begin + (int64_t)t * FS_TILE;
        if (c0 + FS_TILE <= a.Nkv) {
            uint8_t *hb = ring + st * FS_STAGE + which * FS_KT;
            const int64_t nb1 = which ? (int64_t)a.v_nb1 : (int64_t)a.k_nb1;
            const uint8_t *g = (which ? v_head : k_head) + c0 * nb1;
#pragma unroll
            for (int i = 0; i < 16; i++) dma(g + (int64_t)(4 * i) * nb1, which ? voff : koff[i & 3], hb + i * 1024);
        } else {
            issue_clamped(c0, st, which);
        }
    };

    fs_state S;
    fs_init(S);
    const float scale = a.softcap != 0.0f ? a.scale / a.softcap : a.scale;

    // q and this wave's mask values first, then the transfers in the order K0 V0, K1 V1 (when q is in place), then K(t + 2) once the scores of tile t are taken and V(t + 2) once its output
    // is.  All are buffer accesses or ordinary loads: the compiler counts those exactly and waits for q with the transfers in flight.
    const int hr = lane & 3;
    f32x4 qx[2];
    u32x4 mc[MT / 8];
    fs_request_q(a.q, a.q_nb2, hk * R, R, lane, qx);
    fs_request_mask<MT>(a, c_begin, n, lane, mc);
    asm volatile("" ::: "memory");   // the loads are not to be moved behind the transfers
    __builtin_amdgcn_sched_barrier(0);
    {   // without a branch around them (a wave without tiles moves the last one, and waits for it behind the loop): at a join of paths the compiler knows the smaller number of requests in flight only
        const int64_t first = n > 0 ? c_begin : (int64_t)(n_tiles - 1) * FS_TILE;
        issue_clamped(first, 0, 0);
        issue_clamped(first, 0, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    unsigned short *mw = mbuf[wave];
    u32 qv[FS_D / 2];
    fs_spread_q(qx, R, lane, (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)&qbuf[wave][0], qv);
    fs_store_mask<MT>(mc, lane, (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned short *)mw);
    if (!ONE && n > 1) {
        issue(1, 1, 0);
        issue(1, 1, 1);
    }
    // LDS is read and written through inline assembly with waits placed by hand: for an access it can see, the
    // compiler waits for every global-to-LDS transfer in flight, which would serialise the ring.
    // LDS byte addresses of this lane's operands inside a stage
    const unsigned ring_lds = (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)ring;
    const unsigned k_lane = (unsigned)lane * FS_ROW + ((unsigned)(lane & 15) << 4);                      // chunk c at k_lane ^ (c << 4)
    const unsigned v_lane = FS_KT + fs_v_lane(lane);
    const unsigned m_lane = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned short *)mw + (unsigned)lane * 2;
    const unsigned p_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned short *)&pbuf[wave][0][0];
    const unsigned p_wr = p_base + (unsigned)lane * 2, p_rd = p_base + (unsigned)hr * (FS_TILE * 2);

    for (int t = 0; t < n; t++) {
        const int st = ONE ? 0 : t & 1;
        // K(t) has landed when at most V(t), K(t + 1), V(t + 1) are still on their way (transfers complete in the order issued)
        if (!ONE && t + 1 < n) FS_WAIT_VM(48);
        else FS_WAIT_VM(16);
        const unsigned sb = ring_lds + (unsigned)st * FS_STAGE;

        // ---- scores: 16 chunks of this lane's K row, 32 MFMA steps
        u32x4 kc[16];
        u32 mbits;
        asm volatile("ds_read_u16 %0, %1" : "=v"(mbits) : "v"(m_lane + (unsigned)t * (FS_TILE * 2)));
#pragma unroll
        for (int c = 0; c < 16; c++) asm volatile("ds_read_b128 %0, %1" : "=v"(kc[c]) : "v"(sb + (k_lane ^ (unsigned)(c << 4))));
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(mbits), "+v"(kc[0]), "+v"(kc[1]), "+v"(kc[2]), "+v"(kc[3]), "+v"(kc[4]), "+v"(kc[5]), "+v"(kc[6]), "+v"(kc[7]), "+v"(kc[8]), "+v"(kc[9]),
                       "+v"(kc[10]), "+v"(kc[11]), "+v"(kc[12]), "+v"(kc[13]), "+v"(kc[14]), "+v"(kc[15]));
        if (!ONE && t + 2 < n) issue(t + 2, st, 0);   // the K rows are in registers: their half of the stage is free
        fs_scores(qv, kc, half_bits_to_float((unsigned short)mbits), scale, a.softcap, slope, p_wr, S);
        // V(t) has landed when at most K(t + 1), V(t + 1), K(t + 2) are outstanding
        if (!ONE && t + 2 < n) FS_WAIT_VM(48);
        else if (!ONE && t + 1 < n) FS_WAIT_VM(32);
        else FS_WAIT_VM(0);
        fs_output(sb + v_lane, p_rd, S);
        // every LDS read of this stage has returned (the last wait above): the V half may be overwritten
        if (!ONE && t + 2 < n) issue(t + 2, st, 1);
    }
    // a wave without tiles has not waited for its transfers: they must have landed before fs_join takes the ring, and before the wave gives its LDS back
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    if constexpr (ONE) {
        fs_join<NWV>(S, (float *)ring_buf, FS_STAGE / 4, a.ws + ((int64_t)hk * R * a.n_splits + blockIdx.x) * (FS_D + 2), (int64_t)a.n_splits * (FS_D + 2), R, lane, wave);
        return;
    }
    // ---- partial result of this split: un-normalised outputs, running maximum, sum
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (r < R) {
            const float L = wave_sum_dpp(S.lsum[r]);
            float *p = a.ws + (((int64_t)hk * R + r) * a.n_splits + split) * (FS_D + 2);
            p[lane] = S.o0[r];
            p[64 + lane] = S.o1[r];
            if (lane == 0) {
                p[FS_D] = S.m[r];
                p[FS_D + 1] = L;
            }
        }
    }
}

// ---- the same over a Q8_0 / Q4_0 cache in the device row layout --------------------------------------------------------------
// A cell's row in such a cache holds the levels of all its kv heads first and their f16 scales behind them, so the levels of one
// (cell, head) are 128 / 64 contiguous, 16-byte aligned bytes and its four scales 8 bytes: both move by global-to-LDS transfers like
// the f16 rows above (levels 16 bytes per lane, scales 4), half the bytes or less per cell.
// Scores follow the reference's arithmetic for a quantized K (ggml-cpu.c:11037-11046: q is quantized to Q8_0, kq_vec_dot is the
// integer block dot ggml_vec_dot_q8_0_q8_0 / ggml_vec_dot_q4_0_q8_0, ggml-cpu-quants.c): v_mfma_i32_4x4x4_16b_i8 with A = q levels
// (row = head) and B = this lane's cell, one accumulator per 32-element block, then sum_b d_k d_q sumi in f32.
// V (ggml-cpu.c:11078-11090 dequantizes the row and accumulates in f32): the wave turns the tile's levels into d * level as f16 -
// bytes into the low byte of halves whose high byte is 0x64 (1024 + u), minus 1152 or 1032, times the block's scale, all packed
// f16 operations on exact values until the one rounding of the product - and writes them row-major into its own 16 KiB of LDS,
// where fs_output finds what it finds for an f16 cache.
struct fsq_src {
    const uint8_t *lv, *sc;   // levels / scales of (cell 0, kv head 0)
    int64_t head_lv, head_sc; // bytes from one kv head to the next
    int64_t cell_lv, cell_sc; // bytes from one cell to the next
};
template <int T>
struct fsq_geo {
    static constexpr int ROW = T == MI355_Q8_0 ? 128 : 64;   // bytes of levels per (cell, head)
    static constexpr int CH = ROW / 16;                       // 16-byte chunks per row
    static constexpr int RPT = 64 / CH;                       // rows per transfer
    static constexpr int NT = FS_TILE / RPT;                  // level transfers per tile
    static constexpr int CNT = NT + 2;                        // with the two scale transfers
};
constexpr int FSQ_SCALES = FS_TILE * 8;   // bytes of scales per tile and operand

// q of the group's four heads (fs_request_q's eight values per lane) as Q8_0 (quantize_row_q8_0_ref, ggml-quants.c:194-218): qw = the 32 words of levels of head lane % 4,
// through FSQ_QLDS bytes of the wave's LDS; dqa / qsa [head][block] = the f16-rounded scales and the sums of the levels, the same in every lane; zeros past the R heads
constexpr int FSQ_QROW = FS_D + 16, FSQ_QLDS = 4 * FSQ_QROW;
static_assert(FSQ_QLDS <= 32 * FS_ROW, "taken from the room of half a V tile");
__device__ __forceinline__ void fsq_spread_q(f32x4 (&x)[2], int R, int lane, unsigned q_lds, u32 (&qw)[32], float (&dqa)[4][4], int (&qsa)[4][4]) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        x[i >> 2][i & 3] = (lane >> 4) < R ? x[i >> 2][i & 3] : 0.0f;
        amax = fmaxf(amax, fabsf(x[i >> 2][i & 3]));
    }
    amax = lanes_max<4>(amax);   // four lanes hold a block
    float d, id;
    q8_scale(amax, d, id);
    u32x2 w;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        u32 t = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int q = q8_level(x[i][j], id);
            sum += q;
            t |= (u32)(q & 0xFF) << (8 * j);
        }
        w[i] = t;
    }
    sum = lanes_sum_i<4>(sum);
    const float dr = half_bits_to_float(float_to_half_bits(d));
    asm volatile("ds_write_b64 %0, %1" ::"v"(q_lds + (unsigned)(lane >> 4) * FSQ_QROW + (unsigned)(lane & 15) * 8u), "v"(w) : "memory");
    u32x4 t[8];
#pragma unroll
    for (int i = 0; i < 8; i++) asm volatile("ds_read_b128 %0, %1" : "=v"(t[i]) : "v"(q_lds + (unsigned)(lane & 3) * FSQ_QROW + (unsigned)i * 16u));
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            dqa[r][b] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, dr), 16 * r + 4 * b));
            qsa[r][b] = __builtin_amdgcn_readlane(sum, 16 * r + 4 * b);
        }
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]), "+v"(t[4]), "+v"(t[5]), "+v"(t[6]), "+v"(t[7]));
#pragma unroll
    for (int i = 0; i < 8; i++) {
        qw[4 * i] = t[i][0];
        qw[4 * i + 1] = t[i][1];
        qw[4 * i + 2] = t[i][2];
        qw[4 * i + 3] = t[i][3];
    }
}

// raw scores of this lane's cell against the four heads: kc = the chunks of its K row, ksc = its four scales
template <int TK>
__device__ __forceinline__ void fsq_scores(const u32 (&qw)[32], const float (&dqa)[4][4], const int (&qsa)[4][4], const u32x4 (&kc)[fsq_geo<TK>::CH], const u32x2 &ksc,
                                           float (&raw)[4]) {
    i32x4 ab[4];
#pragma unroll
    for (int b = 0; b < 4; b++) ab[b] = i32x4{0, 0, 0, 0};
    if constexpr (TK == MI355_Q8_0) {
#pragma unroll
        for (int c = 0; c < 8; c++)
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const u32 kw = kc[c][w];
                ab[c >> 1] = __builtin_amdgcn_mfma_i32_4x4x4i8((int)qw[4 * c + w], (int)kw, ab[c >> 1], 0, 0, 0);
            }
    } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const u32 kw = kc[c][w];
                ab[c] = __builtin_amdgcn_mfma_i32_4x4x4i8((int)qw[8 * c + w], (int)(kw & 0x0F0F0F0Fu), ab[c], 0, 0, 0);
                ab[c] = __builtin_amdgcn_mfma_i32_4x4x4i8((int)qw[8 * c + 4 + w], (int)((kw >> 4) & 0x0F0F0F0Fu), ab[c], 0, 0, 0);
            }
    }
    float dk[4];
    dk[0] = half_bits_to_float((unsigned short)(ksc[0] & 0xFFFFu));
    dk[1] = half_bits_to_float((unsigned short)(ksc[0] >> 16));
    dk[2] = half_bits_to_float((unsigned short)(ksc[1] & 0xFFFFu));
    dk[3] = half_bits_to_float((unsigned short)(ksc[1] >> 16));
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float sum = 0.0f;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int sumi = TK == MI355_Q8_0 ? ab[b][r] : ab[b][r] - 8 * qsa[r][b];
            sum += (float)sumi * (dk[b] * dqa[r][b]);
        }
        raw[r] = sum;
    }
}

// four bytes u -> the f16 pairs (u0 + bias, u1 + bias) * d and (u2 + bias, u3 + bias) * d; 1024 + u is exact in a half whose high
// byte is 0x64, and so is the sum with bias = -(1024 + offset of the level)
__device__ __forceinline__ u32x2 fsq_bytes_to_f16(u32 u, f16x2 bias, f16x2 d2) {
    const u32 a = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u), b = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const f16x2 x = (__builtin_bit_cast(f16x2, a) + bias) * d2, y = (__builtin_bit_cast(f16x2, b) + bias) * d2;
    return u32x2{__builtin_bit_cast(u32, x), __builtin_bit_cast(u32, y)};
}

// V levels of 32 cells of a stage (LDS byte addresses of the first cell's levels / scales) -> d * level as f16, row-major
// [32][128], at LDS byte address v_f16
template <int TV>
__device__ __forceinline__ void fsq_convert_v(unsigned v_lv, unsigned v_sc, unsigned v_f16, int lane) {
    typedef fsq_geo<TV> G;
    constexpr int NJ = 32 * G::CH / 64;   // chunks per lane: 4 (Q8_0, 16 elements each) or 2 (Q4_0, 32 elements each)
    u32x4 lv[NJ];
    u32 sc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int chunk = j * 64 + lane, row = chunk / G::CH, c = chunk % G::CH;
        const int blk = TV == MI355_Q8_0 ? c >> 1 : c;
        asm volatile("ds_read_b128 %0, %1" : "=v"(lv[j]) : "v"(v_lv + (unsigned)chunk * 16u));
        asm volatile("ds_read_u16 %0, %1" : "=v"(sc[j]) : "v"(v_sc + (unsigned)(row * 8 + blk * 2)));
    }
    if constexpr (NJ == 4)
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(lv[0]), "+v"(lv[1]), "+v"(lv[2]), "+v"(lv[3]), "+v"(sc[0]), "+v"(sc[1]), "+v"(sc[2]), "+v"(sc[3]));
    else
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(lv[0]), "+v"(lv[1]), "+v"(sc[0]), "+v"(sc[1]));
    const f16x2 bias = TV == MI355_Q8_0 ? f16x2{(_Float16)-1152.0f, (_Float16)-1152.0f} : f16x2{(_Float16)-1032.0f, (_Float16)-1032.0f};
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int chunk = j * 64 + lane, row = chunk / G::CH, c = chunk % G::CH;
        const u32 dd = sc[j] | (sc[j] << 16);
        const f16x2 d2 = __builtin_bit_cast(f16x2, dd);
        if constexpr (TV == MI355_Q8_0) {
            // elements 16 c .. 16 c + 7, .. + 15 of the row
            const u32 w0 = lv[j][0], w1 = lv[j][1], w2 = lv[j][2], w3 = lv[j][3];
            const u32x2 e0 = fsq_bytes_to_f16(w0 ^ 0x80808080u, bias, d2), e1 = fsq_bytes_to_f16(w1 ^ 0x80808080u, bias, d2);
            const u32x2 e2 = fsq_bytes_to_f16(w2 ^ 0x80808080u, bias, d2), e3 = fsq_bytes_to_f16(w3 ^ 0x80808080u, bias, d2);
            const u32x4 o0 = {e0[0], e0[1], e1[0], e1[1]}, o1 = {e2[0], e2[1], e3[0], e3[1]};
            const unsigned dst = v_f16 + (unsigned)(row * FS_ROW + c * 32);
            asm volatile("ds_write_b128 %0, %1" ::"v"(dst), "v"(o0) : "memory");
            asm volatile("ds_write_b128 %0, %1 offset:16" ::"v"(dst), "v"(o1) : "memory");
        } else {
            u32x4 o[4];   // elements 32 c + 0..7, 8..15 (low nibbles), 16..23, 24..31 (high nibbles)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const u32 wa = lv[j][2 * h], wb = lv[j][2 * h + 1];
                const u32x2 la = fsq_bytes_to_f16(wa & 0x0F0F0F0Fu, bias, d2), lb = fsq_bytes_to_f16(wb & 0x0F0F0F0Fu, bias, d2);
                const u32x2 ha = fsq_bytes_to_f16((wa >> 4) & 0x0F0F0F0Fu, bias, d2), hb = fsq_bytes_to_f16((wb >> 4) & 0x0F0F0F0Fu, bias, d2);
                o[h] = u32x4{la[0], la[1], lb[0], lb[1]};
                o[2 + h] = u32x4{ha[0], ha[1], hb[0], hb[1]};
            }
            const unsigned dst = v_f16 + (unsigned)(row * FS_ROW + c * 64);
            asm volatile("ds_write_b128 %0, %1" ::"v"(dst), "v"(o[0]) : "memory");
            asm volatile("ds_write_b128 %0, %1 offset:16" ::"v"(dst), "v"(o[1]) : "memory");
            asm volatile("ds_write_b128 %0, %1 offset:32" ::"v"(dst), "v"(o[2]) : "memory");
            asm volatile("ds_write_b128 %0, %1 offset:48" ::"v"(dst), "v"(o[3]) : "memory");
        }
    }
}

// Waves per group (= per compute unit): as many as LDS holds - each wave keeps two stages, half a tile of f16 V, its P^T and the mask
// values of up to FSQ_MAX_TILES tiles.  A wave on its own is one dependent chain (reads, scores, soft-max, conversion, output);
// more of them per compute unit is what keeps its vector ALUs and its transfers busy.
constexpr int FSQ_MAX_TILES = 32;
constexpr int FSQ_VF = 32 * FS_ROW;   // bytes of half a V tile as f16
template <int TK, int TV>
constexpr int fsq_waves() { return TK == MI355_Q8_0 && TV == MI355_Q8_0 ? 3 : (TK == MI355_Q4_0 && TV == MI355_Q4_0 ? 5 : 4); }
static int fsq_waves_rt(int tk, int tv) { return tk == MI355_Q8_0 && tv == MI355_Q8_0 ? 3 : (tk == MI355_Q4_0 && tv == MI355_Q4_0 ? 5 : 4); }
constexpr int FSQ_TOTAL_GROUPS = 256;
// ONE: no wave has more than one tile.  A wave then keeps one stage, LDS holds more of them (of Q8_0 five at 26 KiB each, of Q4_0 eight at 18 KiB), and
// the group's waves join their states, so that the merge launch reads one result per group.  In its place two waves walked two to four tiles
// each: 8192 cells, 32 / 8 heads, Q8_0 16.9 -> 16.2 us, Q4_0 15.9 -> 14.7; 8 / 8 heads 15.7 -> 13.5 and 15.2 -> 13.2; 10240 cells of Q4_0 20.5 -> 16.8.  A result
// per wave costs more than the chain it saves (Q8_0, 8192 cells, 32 / 8: 18.2 us); two waves with a tile or more each lose by joining (4096 cells 13.4 -> 14.3).
template <int TK, int TV>
constexpr int fsq_waves_one() { return TK == MI355_Q8_0 && TV == MI355_Q8_0 ? 5 : (TK == MI355_Q4_0 && TV == MI355_Q4_0 ? 8 : 6); }
static int fsq_waves_one_rt(int tk, int tv) { return tk == MI355_Q8_0 && tv == MI355_Q8_0 ? 5 : (tk == MI355_Q4_0 && tv == MI355_Q4_0 ? 8 : 6); }

template <int TK, int TV, bool ONE>
__global__ void __launch_bounds__(((ONE ? fsq_waves_one<TK, TV>() : fsq_waves<TK, TV>()) * 64), 1) k_fattn_dec_stream_q(fattn_args a, fsq_src ksrc, fsq_src vsrc, int tiles_per_wave, int n_tiles, int R) {
    typedef fsq_geo<TK> GK;
    typedef fsq_geo<TV> GV;
    constexpr int NWV = ONE ? fsq_waves_one<TK, TV>() : fsq_waves<TK, TV>(), STAGES = ONE ? 1 : 2, MT = ONE ? 8 : FSQ_MAX_TILES;
    constexpr int K_LV = FS_TILE * GK::ROW, V_LV = FS_TILE * GV::ROW;
    constexpr int OFF_V = K_LV, OFF_KS = K_LV + V_LV, OFF_VS = OFF_KS + FSQ_SCALES;
    constexpr int STAGE = OFF_VS + FSQ_SCALES;
    constexpr int CK = GK::CNT, CV = GV::CNT;   // transfers of the K / V part of a tile
    __shared__ __attribute__((aligned(1024))) uint8_t ring_buf[NWV * STAGES * STAGE];
    __shared__ __attribute__((aligned(1024))) uint8_t vf_buf[NWV * FSQ_VF];   // half of the wave's V tile as f16
    __shared__ __attribute__((aligned(16))) unsigned short pbuf[NWV][4][FS_TILE];
    __shared__ __attribute__((aligned(16))) unsigned short mbuf[NWV][MT * FS_TILE];
    asm volatile("" ::"v"((void *)ring_buf), "v"((void *)vf_buf) : "memory");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int split = (int)blockIdx.x * (int)(blockDim.x >> 6) + wave;   // the launch may give a group fewer than NWV waves
    const int64_t hk = blockIdx.y;
    const int t_begin = split * tiles_per_wave;
    const int t_end = t_begin + tiles_per_wave < n_tiles ? t_begin + tiles_per_wave : n_tiles;
    const int n = t_end > t_begin ? t_end - t_begin : 0;
    const int64_t c_begin = (int64_t)t_begin * FS_TILE;

    float slope[4];
    fs_slopes(a, hk * R, slope);
    uint8_t *ring = ring_buf + wave * (STAGES * STAGE);
    const uint8_t *k_lv = ksrc.lv + hk * ksrc.head_lv, *k_sc = ksrc.sc + hk * ksrc.head_sc;
    const uint8_t *v_lv = vsrc.lv + hk * vsrc.head_lv, *v_sc = vsrc.sc + hk * vsrc.head_sc;
    // per-lane offsets of the transfers.  K levels: transfer i moves rows RPT i .. + RPT - 1, lane p -> row RPT i + p / CH, LDS position
    // p % CH, which holds chunk position ^ swz(row) (swz: (row >> 1) & 7 for 128-byte rows, (row >> 2) & 3 for 64-byte rows), so that
    // the 64 lanes reading chunk c of their own rows hit all banks.  V levels: rows as they are.  Scales: two transfers of 32 rows.
    unsigned koff[2], voff, ksoff, vsoff;
    {
        const unsigned p = (unsigned)lane;
        if constexpr (TK == MI355_Q8_0) {
#pragma unroll
            for (int e = 0; e < 2; e++) koff[e] = (p >> 3) * (unsigned)ksrc.cell_lv + (((p & 7) ^ ((4 * e + (p >> 4)) & 7)) << 4);
        } else {
            koff[0] = koff[1] = (p >> 2) * (unsigned)ksrc.cell_lv + (((p & 3) ^ ((p >> 4) & 3)) << 4);
        }
        voff = TV == MI355_Q8_0 ? (p >> 3) * (unsigned)vsrc.cell_lv + ((p & 7) << 4) : (p >> 2) * (unsigned)vsrc.cell_lv + ((p & 3) << 4);
        ksoff = (p >> 1) * (unsigned)ksrc.cell_sc + ((p & 1) << 2);
        vsoff = (p >> 1) * (unsigned)vsrc.cell_sc + ((p & 1) << 2);
    }
    auto dma16 = [&](const uint8_t *g, unsigned off, uint8_t *l) {   // g, l: wave-uniform
        buf_to_lds16(g, off, 0, l);
    };
    auto dma4 = [&](const uint8_t *g, unsigned off, uint8_t *l) { buf_to_lds4(g, off, 0, l); };
    // which = 0: K levels and scales into stage st (CK transfers), 1: V (CV transfers).  The cell they start at; rows past the end of the cache repeat the last cell (their
    // scores are discarded)
    auto issue_clamped = [&](int64_t c0, int st, int which) {
        uint8_t *sb = ring + st * STAGE;
        const int64_t nb_lv = which ? vsrc.cell_lv : ksrc.cell_lv, nb_sc = which ? vsrc.cell_sc : ksrc.cell_sc;
        const uint8_t *g = (which ? v_lv : k_lv) + c0 * nb_lv, *gs = (which ? v_sc : k_sc) + c0 * nb_sc;
        uint8_t *l_lv = sb + (which ? OFF_V : 0), *l_sc = sb + (which ? OFF_VS : OFF_KS);
        const int NT = which ? GV::NT : GK::NT, RPT = which ? GV::RPT : GK::RPT, CH = which ? GV::CH : GK::CH;
        const int last = a.Nkv - c0 < FS_TILE ? (int)(a.Nkv - 1 - c0) : FS_TILE - 1;
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (i < NT) {
                const int row = RPT * i + lane / CH, pos = lane % CH;
                const int swz = which ? 0 : (TK == MI355_Q8_0 ? (row >> 1) & 7 : (row >> 2) & 3);
                dma16(g, (unsigned)(row < last ? row : last) * (unsigned)nb_lv + (unsigned)((pos ^ swz) << 4), l_lv + i * 1024);
            }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = 32 * i + (lane >> 1);
            dma4(gs, (unsigned)(row < last ? row : last) * (unsigned)nb_sc + (unsigned)((lane & 1) << 2), l_sc + i * 256);
        }
    };
    auto issue = [&](int t, int st, int which) {
        const int64_t c0 = c_begin + (int64_t)t * FS_TILE;
        if (c0 + FS_TILE <= a.Nkv) {
            uint8_t *sb = ring + st * STAGE;
            const int64_t nb_lv = which ? vsrc.cell_lv : ksrc.cell_lv, nb_sc = which ? vsrc.cell_sc : ksrc.cell_sc;
            uint8_t *l_lv = sb + (which ? OFF_V : 0), *l_sc = sb + (which ? OFF_VS : OFF_KS);
            const int NT = which ? GV::NT : GK::NT, RPT = which ? GV::RPT : GK::RPT;
            const uint8_t *g = (which ? v_lv : k_lv) + c0 * nb_lv, *gs = (which ? v_sc : k_sc) + c0 * nb_sc;
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (i < NT) dma16(g + (int64_t)(RPT * i) * nb_lv, which ? voff : koff[i & 1], l_lv + i * 1024);
            dma4(gs, which ? vsoff : ksoff, l_sc);
            dma4(gs + 32 * nb_sc, which ? vsoff : ksoff, l_sc + 256);
        } else {
            issue_clamped(c0, st, which);
        }
    };

    fs_state S;
    fs_init(S);
    const float scale = a.softcap != 0.0f ? a.scale / a.softcap : a.scale;
    // q and this wave's mask values first, the transfers of the first tile behind them (see k_fattn_dec_stream)
    const int hr = lane & 3;
    f32x4 qx[2];
    u32x4 mc[MT / 8];
    fs_request_q(a.q, a.q_nb2, hk * R, R, lane, qx);
    fs_request_mask<MT>(a, c_begin, n, lane, mc);
    asm volatile("" ::: "memory");   // the loads are not to be moved behind the transfers
    __builtin_amdgcn_sched_barrier(0);
    {
        const int64_t first = n > 0 ? c_begin : (int64_t)(n_tiles - 1) * FS_TILE;
        issue_clamped(first, 0, 0);
        issue_clamped(first, 0, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    unsigned short *mw = mbuf[wave];
    u32 qw[32];
    float dqa[4][4];
    int qsa[4][4];
    fsq_spread_q(qx, R, lane, (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)(vf_buf + wave * FSQ_VF), qw, dqa, qsa);   // no V there yet
    fs_store_mask<MT>(mc, lane, (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned short *)mw);
    if (!ONE && n > 1) {
        issue(1, 1, 0);
        issue(1, 1, 1);
    }
    // LDS is read and written through inline assembly with waits placed by hand (see k_fattn_dec_stream).
    const unsigned ring_lds = (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)ring;
    const unsigned vf_lds = (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)(vf_buf + wave * FSQ_VF);
    const unsigned k_lane = TK == MI355_Q8_0 ? (unsigned)lane * 128u + ((((unsigned)lane >> 1) & 7u) << 4) : (unsigned)lane * 64u + ((((unsigned)lane >> 2) & 3u) << 4);
    const unsigned m_lane = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned short *)mw + (unsigned)lane * 2;
    const unsigned p_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned short *)&pbuf[wave][0][0];
    const unsigned p_wr = p_base + (unsigned)lane * 2, p_rd = p_base + (unsigned)hr * (FS_TILE * 2);

    for (int t = 0; t < n; t++) {
        const int st = ONE ? 0 : t & 1;
        // K(t) has landed when at most V(t), K(t + 1), V(t + 1) are still on their way (transfers complete in the order issued)
        if (!ONE && t + 1 < n) FS_WAIT_VM(CV + CK + CV);
        else FS_WAIT_VM(CV);
        const unsigned sb = ring_lds + (unsigned)st * STAGE;
        u32x4 kc[GK::CH];
        u32x2 ksc;
        u32 mbits;
        asm volatile("ds_read_u16 %0, %1" : "=v"(mbits) : "v"(m_lane + (unsigned)t * (FS_TILE * 2)));
        asm volatile("ds_read_b64 %0, %1" : "=v"(ksc) : "v"(sb + (unsigned)OFF_KS + (unsigned)lane * 8u));
#pragma unroll
        for (int c = 0; c < GK::CH; c++) asm volatile("ds_read_b128 %0, %1" : "=v"(kc[c]) : "v"(sb + (k_lane ^ (unsigned)(c << 4))));
        if constexpr (GK::CH == 8)
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(mbits), "+v"(ksc), "+v"(kc[0]), "+v"(kc[1]), "+v"(kc[2]), "+v"(kc[3]), "+v"(kc[4]), "+v"(kc[5]), "+v"(kc[6]), "+v"(kc[7]));
        else
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(mbits), "+v"(ksc), "+v"(kc[0]), "+v"(kc[1]), "+v"(kc[2]), "+v"(kc[3]));
        if (!ONE && t + 2 < n) issue(t + 2, st, 0);   // the K rows are in registers: their part of the stage is free
        float raw[4];
        fsq_scores<TK>(qw, dqa, qsa, kc, ksc, raw);
        fs_softmax(raw, half_bits_to_float((unsigned short)mbits), scale, a.softcap, slope, p_wr, S);
        // V(t) has landed when at most K(t + 1), V(t + 1), K(t + 2) are outstanding
        if (!ONE && t + 2 < n) FS_WAIT_VM(CK + CV + CK);
        else if (!ONE && t + 1 < n) FS_WAIT_VM(CK + CV);
        else FS_WAIT_VM(0);
        // the tile's V in two halves of 32 cells through the wave's 8 KiB of f16 rows
        fsq_convert_v<TV>(sb + (unsigned)OFF_V, sb + (unsigned)OFF_VS, vf_lds, lane);
        fs_output<8>(vf_lds + fs_v_lane(lane), p_rd, S);
        fsq_convert_v<TV>(sb + (unsigned)(OFF_V + 32 * GV::ROW), sb + (unsigned)(OFF_VS + 32 * 8), vf_lds, lane);
        // the levels are in registers or already converted: the V part of the stage may be overwritten
        if (!ONE && t + 2 < n) issue(t + 2, st, 1);
        fs_output<8>(vf_lds + fs_v_lane(lane), p_rd + 64, S);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the transfers of a wave without tiles (see k_fattn_dec_stream)

    if constexpr (ONE) {
        fs_join<NWV>(S, (float *)vf_buf, FSQ_VF / 4, a.ws + ((int64_t)hk * R * a.n_splits + blockIdx.x) * (FS_D + 2), (int64_t)a.n_splits * (FS_D + 2), R, lane, wave);
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (r < R) {
            const float L = wave_sum_dpp(S.lsum[r]);
            float *p = a.ws + (((int64_t)hk * R + r) * a.n_splits + split) * (FS_D + 2);
            p[lane] = S.o0[r];
            p[64 + lane] = S.o1[r];
            if (lane == 0) {
                p[FS_D] = S.m[r];
                p[FS_D + 1] = L;
            }
        }
    }
}

// ---- short caches: at most 512 cells, one launch -------------------------------------------------------------------------------
// One wave per 64-cell tile (up to eight).  Nothing here is bound by bytes: the time is one trip to memory plus the arithmetic of one tile, so a wave requests
// everything at once - its K and V tiles as coalesced 16-byte loads into registers (four whole rows per instruction), q, its mask value - and then passes first K, then V
// through its own 16 KiB of LDS to bring them into operand form: K rows with their chunks XOR-ed across the banks, so that each lane reads back the row of its
// cell; V row-major for the transposing reads.  (A lane loading its own K row directly would touch 64 cache lines per instruction: measured 2.8 us per wave of the group.)
// The waves' states meet in LDS; the group normalises and writes the output (and its Q8_1 form where the next product wants it), so no second launch merges anything.
// As many groups per kv head as leave one on every compute unit (a group takes one's LDS), with the same bits: all form the scores of their heads over all cells.
//   PARTS = 2: a group for each half of the output elements, which reads only its half of every V row.  In a model the cache comes from HBM and a compute unit's own requests take
//     their time: 512 cells are 256 KiB for one group per kv head, 192 KiB for one of two (K reaches the second one through L2).
//   NH: query heads of a group.  The soft-max of a head is some 90 instructions of each wave.
// 32 / 8 heads, 512 cells, us: one group per kv head 7.6, two 6.3, four (NH = 2) 5.9, eight (NH = 1) 5.8; 288 cells 7.1, 5.7, 5.2, 5.1.  A group too many costs a second round: 160 / 40 heads,
// 512 cells 11.1 with NH = 1, 6.8 with 2, 7.4 with 4; 256 / 64 heads 11.2, 6.8, 7.4.  With 32-bit offsets and arguments in registers, a layer of the 8B model 45.9 -> 45.2, with one
// head per group 44.3 (a token 1553 -> 1508).
//   P32: up to FSS_P32_CELLS cells, where the vector kernel, with f32 probabilities and masked cells not read, is the other choice: probabilities as f32 on the vector units (fs_output_f32),
//     V of masked cells as zeros, scores in more and shorter chains.  (Probabilities as the sum of two f16 values on the f16 matrix instruction gave NaN for an infinite value of a visible
//     cell - zero or a negative remainder times infinity - and lost the lower bits of weights below 2^-14: 1.6e-4 of an output that weights of 2^-20 .. 2^-30 make, 3e-6 as f32.)  Relative
//     error against 64 bits, 2-norm, 32 .. 256 cells: 1.1e-7 .. 1.9e-7, the vector kernel's 1.2e-7 .. 1.9e-7.  The vector kernel exchanges each score between sixteen lanes; 32 / 8 heads,
//     32 / 128 / 256 cells, us: 4.5, 4.7, 5.6 there, 3.7, 3.9, 4.7 here; 512 / 128 heads 7.1, 7.2, 10.8 and 4.7, 6.0, 7.5.
constexpr int FSS_MAX_WAVES = 8, FSS_P32_WAVES = 4, FSS_P32_CELLS = FSS_P32_WAVES * FS_TILE;

// The arguments ahead of `a` are all that the requests need, and in registers when a wave starts (fourteen words): read from `a` they are two trips to memory, the second
// behind the mask's.  cells: Nkv and, from bit 16, R.  A tile's rows are less than 2^30 bytes apart: 32-bit offsets from one scalar address per wave.
template <int PARTS, int NH, bool P32>
__global__ void __launch_bounds__((P32 ? FSS_P32_WAVES : FSS_MAX_WAVES) * 64, P32 ? 2 : 1) k_fattn_dec_short(const uint8_t *__restrict__ q, const uint8_t *__restrict__ k, const uint8_t *__restrict__ v,
                                                                           const uint8_t *__restrict__ mask, u32 q_nb2, u32 k_nb1, u32 k_nb2, u32 v_nb1, u32 v_nb2, u32 cells,
                                                                           fattn_args a) {
    static_assert(PARTS == 2 || (PARTS == 1 && !P32), "whole rows of V or halves");
    constexpr int MAXW = P32 ? FSS_P32_WAVES : FSS_MAX_WAVES, PSZ = P32 ? NH * 4 : 4 * 2;   // PSZ: bytes of probabilities per cell
    constexpr int DO = FS_D / PARTS, VIT = 16 / PARTS, VCH = 16 / PARTS;   // output elements of the group; V loads; 16-byte chunks of V per row
    __shared__ __attribute__((aligned(1024))) uint8_t tbuf[MAXW * FS_KT];
    __shared__ __attribute__((aligned(16))) uint8_t pbuf[MAXW][FS_TILE * PSZ];
    __shared__ float s_m[MAXW][NH], s_l[MAXW][NH];
    __shared__ float s_o[MAXW][NH][DO];
    __shared__ __attribute__((aligned(16))) uint8_t qbuf[MAXW][FS_QLDS];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t hk = blockIdx.x;
    const int part = (int)blockIdx.y;   // PARTS == 2: elements 64 part .. + 63 of the output
    const int Nkv = (int)(cells & 0xFFFF), HR = (int)(cells >> 16), n_waves = (Nkv + FS_TILE - 1) / FS_TILE;
    const int64_t head0 = hk * HR + NH * (int)blockIdx.z;
    const int R = HR - NH * (int)blockIdx.z < NH ? HR - NH * (int)blockIdx.z : NH;   // heads of the group
    const int c0 = wave * FS_TILE, last = Nkv - 1 - c0;   // last: the last cell from the tile's first
    const int rsub = lane >> 4, pos = lane & 15;

    // q of the group's heads (two coalesced loads per lane) and the mask value first, K and V behind them: loads return in the order of their issue
    f32x4 qx[2];
    fs_request_q(q, q_nb2, head0, R, lane, qx);
    // (without a mask some word of q is read in its place: at a join of two paths the compiler would wait for everything)
    const unsigned short *mrow = (const unsigned short *)(mask ? mask : q);
    unsigned short mbits = mrow[!mask ? 0 : c0 + (lane < last ? lane : last)];
    __builtin_amdgcn_sched_barrier(0);
    // load i: rows 4i .. 4i + 3, lane -> row 4i + lane / 16, chunk lane % 16 (rows past the end repeat the last cell; their weights are zero)
    // (half rows of V: rows 8i .. 8i + 7, lane -> row 8i + lane / 8, chunk lane % 8 of the half)
    const int vsub = lane / VCH, vpos = lane % VCH + VCH * part;
    u32x4 kraw[16], vraw[VIT];
    const uint8_t *kt = k + hk * (uint64_t)k_nb2 + (uint64_t)c0 * k_nb1, *vt = v + hk * (uint64_t)v_nb2 + (uint64_t)c0 * v_nb1;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int row = 4 * i + rsub < last ? 4 * i + rsub : last;
        kraw[i] = load16(kt + (__umul24((u32)row, k_nb1) + (u32)(pos << 4)));
    }
#pragma unroll
    for (int i = 0; i < VIT; i++) {
        const int at = (64 / VIT) * i + vsub, row = at < last ? at : last;
        vraw[i] = load16(vt + (__umul24((u32)row, v_nb1) + (u32)(vpos << 4)));
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!mask) mbits = 0;
    if (lane > last) mbits = 0xFC00;   // -inf
    float slope[4];
    fs_slopes(a, head0, slope);
    const float scale = a.softcap != 0.0f ? a.scale / a.softcap : a.scale;
    u32 qv[FS_D / 2];
    fs_spread_q(qx, R, lane, (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)&qbuf[wave][0], qv);

    // K through LDS: chunk c of row r at position c ^ (r & 15); then each lane reads the row of its cell
    uint8_t *tb = tbuf + wave * FS_KT;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int row = 4 * i + rsub;
        *(u32x4 *)(tb + row * FS_ROW + ((pos ^ (row & 15)) << 4)) = kraw[i];
    }
    u32x4 kc[16];
#pragma unroll
    for (int c = 0; c < 16; c++) kc[c] = *(const u32x4 *)(tb + lane * FS_ROW + ((c ^ (lane & 15)) << 4));

    fs_state S;
    fs_init(S);
    const unsigned p_base = (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)&pbuf[wave][0];
    fs_scores<NH, P32>(qv, kc, half_bits_to_float(mbits), scale, a.softcap, slope, p_base + (unsigned)lane * (P32 ? 4 : 2), S);

    // V through the same bytes, row-major (the K rows are in registers).  P32: zeros for masked cells, whatever they hold: their weight of zero would not hide an infinity
    const uint64_t in_use = __ballot(half_bits_to_float(mbits) != -INFINITY);
#pragma unroll
    for (int i = 0; i < VIT; i++) {
        if constexpr (P32)
            if (!((in_use >> ((64 / VIT) * i + vsub)) & 1)) vraw[i] = u32x4{0, 0, 0, 0};
        *(u32x4 *)(tb + ((64 / VIT) * i + vsub) * FS_ROW + (vpos << 4)) = vraw[i];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // fs_output reads LDS through inline assembly: nothing may be moved across
    const unsigned v_addr = (unsigned)(uintptr_t)(void __attribute__((address_space(3))) *)tb + fs_v_lane(lane), p_rd = p_base + (unsigned)(lane & 3) * (FS_TILE * 2);
    if constexpr (P32)
        fs_output_f32<NH>((const uint8_t __attribute__((address_space(3))) *)(uintptr_t)(v_addr + (unsigned)(part * 128)), (const float __attribute__((address_space(3))) *)(uintptr_t)p_base, lane, S.o0);
    else if constexpr (PARTS == 1) fs_output(v_addr, p_rd, S);
    else if (part == 0) fs_output_half<0>(v_addr, p_rd, S.o0);   // uniform
    else fs_output_half<1>(v_addr, p_rd, S.o0);

    // ---- the waves' states meet in LDS
#pragma unroll
    for (int r = 0; r < NH; r++) {
        const float L = wave_sum_dpp(S.lsum[r]);
        if (lane == 0) {
            s_m[wave][r] = S.m[r];
            s_l[wave][r] = L;
        }
        s_o[wave][r][lane] = S.o0[r];
        if constexpr (PARTS == 1) s_o[wave][r][64 + lane] = S.o1[r];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < R * DO; idx += n_waves * 64) {   // whole waves: R * DO and the group size are multiples of 64
        const int r = idx / DO, d = idx % DO;
        float M = s_m[0][r];
        for (int w = 1; w < n_waves; w++) M = fmaxf(M, s_m[w][r]);
        float L = 0.0f, O = 0.0f;
        for (int w = 0; w < n_waves; w++) {
            const float f = __expf(s_m[w][r] - M);
            L += s_l[w][r] * f;
            O += s_o[w][r][d] * f;
        }
        const int64_t head = head0 + r;
        const float o = O / L;
        const int64_t at = head * FS_D + 64 * part + d;
        a.dst[at] = o;
        if (a.act_q) quantize_lane32(o, a.act_q, a.act_s, at);
    }
}

int launch_fattn_dec_short(hipStream_t s, fattn_args &a, int64_t D) {
    const int64_t R = a.Hq / a.Hkv;
    if (D != FS_D || a.Nq != 1 || R > 4 || a.Hkv > 65535 || a.Nkv > FSS_MAX_WAVES * FS_TILE) return 1;
    if ((a.q_nb2 % 16) != 0 || (a.k_nb1 % 16) != 0 || (a.k_nb2 % 16) != 0 || (a.v_nb1 % 16) != 0 || (a.v_nb2 % 16) != 0) return 1;
    if (a.k_nb1 >> 24 || a.v_nb1 >> 24 || a.q_nb2 >> 32 || a.k_nb2 >> 32 || a.v_nb2 >> 32) return 1;   // the kernel's offsets
    constexpr int64_t CU = 256;   // compute units
    const int n_waves = (int)((a.Nkv + FS_TILE - 1) / FS_TILE);
#define MI355_FSS_ARGS dim3((unsigned)n_waves * 64), 0, s, a.q, a.k, a.v, a.mask, (u32)a.q_nb2, (u32)a.k_nb1, (u32)a.k_nb2, (u32)a.v_nb1, (u32)a.v_nb2, (u32)a.Nkv | (u32)R << 16, a
#define MI355_FSS_LAUNCH(P32, RES)                                                                                                                                        \
    if (2 * a.Hq <= RES) MI355_LAUNCH((k_fattn_dec_short<2, 1, P32>), dim3((unsigned)a.Hkv, 2, (unsigned)R), MI355_FSS_ARGS);                                              \
    else if (2 * a.Hkv * ((R + 1) / 2) <= RES) MI355_LAUNCH((k_fattn_dec_short<2, 2, P32>), dim3((unsigned)a.Hkv, 2, (unsigned)((R + 1) / 2)), MI355_FSS_ARGS);            \
    else if (2 * a.Hkv <= RES) MI355_LAUNCH((k_fattn_dec_short<2, 4, P32>), dim3((unsigned)a.Hkv, 2), MI355_FSS_ARGS);
    if (a.Nkv <= FSS_P32_CELLS) {
        // two groups of this form share a compute unit's LDS, which pays for groups of one wave: 195 / 65 heads, 64 cells 5.2 -> 4.5 us, 512 / 128 heads 5.4 -> 4.8; with more waves not
        // (160 / 40 heads, 128 cells 4.6 -> 4.8, 256 cells 5.6 -> 6.5)
        MI355_FSS_LAUNCH(true, (a.Nkv <= FS_TILE ? 2 * CU : CU))
        else return 1;
    } else {
        MI355_FSS_LAUNCH(false, CU)
        else MI355_LAUNCH((k_fattn_dec_short<1, 4, false>), dim3((unsigned)a.Hkv), MI355_FSS_ARGS);
    }
#undef MI355_FSS_LAUNCH
#undef MI355_FSS_ARGS
    return launch_status("k_fattn_dec_short");
}

// One query token, head size 128, R <= 4 query heads per kv head, rows 16-byte aligned.  Sets a.n_splits; the caller merges the
// splits with k_fattn_combine.  Returns 1 when the shape is not served.
int launch_fattn_dec_stream(hipStream_t s, fattn_args &a, int64_t D, size_t ws_bytes) {
    const int64_t R = a.Hq / a.Hkv;
    if (D != FS_D || a.Nq != 1 || R > 4 || a.Hkv > 65535 || a.ws == nullptr) return 1;
    if ((a.q_nb2 % 16) != 0 || (a.k_nb1 % 16) != 0 || (a.k_nb2 % 16) != 0 || (a.v_nb1 % 16) != 0 || (a.v_nb2 % 16) != 0) return 1;
    if (a.k_nb1 >= ((size_t)1 << 26) || a.v_nb1 >= ((size_t)1 << 26)) return 1;   // the transfers' per-lane offsets are 32-bit
    const int64_t n_tiles = (a.Nkv + FS_TILE - 1) / FS_TILE;
    int64_t waves_per_head = FS_TOTAL_WAVES / a.Hkv;
    if (waves_per_head < FS_WAVES) waves_per_head = FS_WAVES;
    if (waves_per_head > 256) waves_per_head = 256;   // k_fattn_combine takes up to 256 splits
    int64_t tiles_per_wave = (n_tiles + waves_per_head - 1) / waves_per_head;
    if (tiles_per_wave > FS_MAX_TILES) return 1;
    int64_t n_splits = (n_tiles + tiles_per_wave - 1) / tiles_per_wave;
    n_splits = (n_splits + FS_WAVES - 1) / FS_WAVES * FS_WAVES;   // whole groups; a wave without tiles writes an empty partial
    // a tile per wave where one group of up to four waves per compute unit holds them all
    const int64_t one_wv = (n_tiles * a.Hkv + FS_TOTAL_WAVES / FS_WAVES - 1) / (FS_TOTAL_WAVES / FS_WAVES), one_groups = (n_tiles + one_wv - 1) / one_wv;
    const bool one = tiles_per_wave > 1 && one_wv <= FS_WAVES_ONE && one_groups <= n_splits;
    if (one) n_splits = one_groups;
    if (ws_bytes < (size_t)a.Hq * (size_t)n_splits * (size_t)(FS_D + 2) * sizeof(float)) return 1;
    a.n_splits = (int)n_splits;
    if (one) MI355_LAUNCH(k_fattn_dec_stream<true>, dim3((unsigned)n_splits, (unsigned)a.Hkv), dim3((unsigned)one_wv * 64), 0, s, a, 1, (int)n_tiles, (int)R);
    else MI355_LAUNCH(k_fattn_dec_stream<false>, dim3((unsigned)(n_splits / FS_WAVES), (unsigned)a.Hkv), dim3(FS_WAVES * 64), 0, s, a, (int)tiles_per_wave, (int)n_tiles, (int)R);
    return launch_status("k_fattn_dec_stream");
}

// fsq_src of a kv_src in the device row layout; false when the operand does not have the shape the kernel moves (whole heads of four
// blocks inside one row of the owner, levels 16-byte and scales 4-byte aligned)
static bool fsq_describe(int type, const kv_src &q, fsq_src &o) {
    if (q.row_blocks <= 0 || q.base == nullptr) return false;
    const int64_t BB = type == MI355_Q8_0 ? Q8_0_BYTES : Q4_0_BYTES, LB = type == MI355_Q8_0 ? 32 : 16;
    const int64_t row0 = q.first_block / q.row_blocks, b0 = q.first_block % q.row_blocks, RB = q.row_blocks * BB;
    if (q.head_blocks < FS_D / 32) return false;   // (that heads and cells stay inside their rows of the owner was checked with kv_src)
    o.lv = q.base + row0 * RB + b0 * LB;
    o.sc = q.base + row0 * RB + q.row_blocks * LB + b0 * 2;
    o.head_lv = q.head_blocks * LB;
    o.head_sc = q.head_blocks * 2;
    o.cell_lv = q.cell_lv;
    o.cell_sc = q.cell_sc;
    if (((uintptr_t)o.lv & 15) != 0 || (o.head_lv & 15) != 0 || (o.cell_lv & 15) != 0 || ((uintptr_t)o.sc & 3) != 0 || (o.head_sc & 3) != 0 || (o.cell_sc & 3) != 0) return false;
    if (o.cell_lv >= ((int64_t)1 << 26) || o.cell_sc >= ((int64_t)1 << 26)) return false;   // the per-lane offsets are 32-bit
    return true;
}

// Groups per kv head of `waves` tiles each; with empty ones to whole turns of the eight XCDs where that leaves one group per compute unit, so that a group's range of
// cells is on one XCD whatever the head: Q4_0, 32 / 8 heads, device us, 9216 cells 29 groups 20.1, 32 16.7 (two to four tiles per wave 18.4); 11776 cells 31
// groups 21.9, 32 18.5 (21.2).  (Not over f16, whose rows are whole lines: 24 / 8 heads, 5120 cells 12.3 / 13.2.)  most: what the workspace rule allows
static int64_t fsq_one_groups(int64_t n_tiles, int64_t waves, int64_t Hkv, int64_t most) {
    const int64_t n = (n_tiles + waves - 1) / waves, whole = (n + 7) / 8 * 8;
    return whole * Hkv <= FSQ_TOTAL_GROUPS && whole <= most ? whole : n;
}

// One query token over a long Q8_0 / Q4_0 cache in the device row layout (a.type_k, a.type_v, a.kq, a.vq filled in), head size 128,
// R <= 4.  Sets a.n_splits; the caller merges the splits with k_fattn_combine.  Returns 1 when the shape is not served.
int launch_fattn_dec_stream_q(hipStream_t s, fattn_args &a, int64_t D, size_t ws_bytes) {
    const int64_t R = a.Hq / a.Hkv;
    if (D != FS_D || a.Nq != 1 || R > 4 || a.Hkv > 65535 || a.ws == nullptr || (a.q_nb2 % 16) != 0) return 1;
    if ((a.type_k != MI355_Q8_0 && a.type_k != MI355_Q4_0) || (a.type_v != MI355_Q8_0 && a.type_v != MI355_Q4_0)) return 1;
    fsq_src ks, vs;
    if (!fsq_describe(a.type_k, a.kq, ks) || !fsq_describe(a.type_v, a.vq, vs)) return 1;
    const int64_t n_tiles = (a.Nkv + FS_TILE - 1) / FS_TILE;
    // Waves per group: all that LDS holds once every wave has a dozen tiles or more (131072 cells of 8 kv heads: 94.5 -> 82 us for
    // Q8_0, 90 -> 73 us for Q4_0); with fewer tiles, two per group spread over more compute units are quicker (32768 cells: 34 us
    // against 39 us).
    int nwv = fsq_waves_rt(a.type_k, a.type_v);
    if (n_tiles * a.Hkv < (int64_t)FSQ_TOTAL_GROUPS * nwv * 12) nwv = 2;
    int64_t waves_per_head = (int64_t)FSQ_TOTAL_GROUPS * nwv / a.Hkv;
    if (waves_per_head < nwv) waves_per_head = nwv;
    if (waves_per_head > 256) waves_per_head = 256;   // k_fattn_combine takes up to 256 splits
    int64_t tiles_per_wave = (n_tiles + waves_per_head - 1) / waves_per_head;
    if (tiles_per_wave > FSQ_MAX_TILES) return 1;
    int64_t n_splits = (n_tiles + tiles_per_wave - 1) / tiles_per_wave;
    n_splits = (n_splits + nwv - 1) / nwv * nwv;   // whole groups; a wave without tiles writes an empty partial
    // A tile per wave where one group per compute unit holds them all.  Five waves of Q8_0 only for up to two query heads per kv head (10240 cells,
    // 16 / 8 heads 19.4 -> 18.2 us, 32 / 8 heads 20.35 -> 20.45).
    bool one = false;
    const int64_t one_wv = (n_tiles * a.Hkv + FSQ_TOTAL_GROUPS - 1) / FSQ_TOTAL_GROUPS, one_groups = fsq_one_groups(n_tiles, one_wv, a.Hkv, n_splits);
    const int one_max = a.type_k == MI355_Q8_0 && a.type_v == MI355_Q8_0 && R > 2 ? 4 : fsq_waves_one_rt(a.type_k, a.type_v);
    if (tiles_per_wave > 1 && one_wv <= one_max && one_groups <= n_splits) {
        one = true;
        nwv = (int)one_wv;
        tiles_per_wave = 1;
        n_splits = one_groups;
    }
    if (n_splits > 256) return 1;
    if (ws_bytes < (size_t)a.Hq * (size_t)n_splits * (size_t)(FS_D + 2) * sizeof(float)) return 1;
    a.n_splits = (int)n_splits;
    const dim3 grid((unsigned)(one ? n_splits : n_splits / nwv), (unsigned)a.Hkv), block((unsigned)nwv * 64);
#define MI355_FSQ_LAUNCH(TK, TV) \
    do { \
        if (one) MI355_LAUNCH((k_fattn_dec_stream_q<TK, TV, true>), grid, block, 0, s, a, ks, vs, 1, (int)n_tiles, (int)R); \
        else MI355_LAUNCH((k_fattn_dec_stream_q<TK, TV, false>), grid, block, 0, s, a, ks, vs, (int)tiles_per_wave, (int)n_tiles, (int)R); \
    } while (0)
    if (a.type_k == MI355_Q8_0 && a.type_v == MI355_Q8_0) MI355_FSQ_LAUNCH(MI355_Q8_0, MI355_Q8_0);
    else if (a.type_k == MI355_Q8_0) MI355_FSQ_LAUNCH(MI355_Q8_0, MI355_Q4_0);
    else if (a.type_v == MI355_Q8_0) MI355_FSQ_LAUNCH(MI355_Q4_0, MI355_Q8_0);
    else MI355_FSQ_LAUNCH(MI355_Q4_0, MI355_Q4_0);
#undef MI355_FSQ_LAUNCH
    return launch_status("k_fattn_dec_stream_q");
}

}  // namespace mi355
