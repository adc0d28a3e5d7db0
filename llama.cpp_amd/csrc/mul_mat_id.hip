// MUL_MAT_ID host entry: quantize the nb1*T rows of b once, then route every
// (token, expert slot) pair to its expert's weights on the device: per-slot GEMV for a few slots,
// the weight-streaming kernel for a few per expert, slots sorted by expert and one tile launch over all experts for many.
#include "common.hpp"
#include "qdot.hpp"

#include <math.h>

using namespace mi355;

extern "C" {

// From this many (token, expert slot) pairs on the slots may be sorted by expert and run through the routed tile kernels, which read every
// expert's matrix once; with fewer each slot streams its expert's matrix through the GEMV.  use_skinny takes calls from both.
static constexpr int64_t ROUTED_MIN_SLOTS = 32;   // measured cross-over on 8 experts of 14336 x 4096

static bool use_routed_tiles(int type, const void *as, int64_t N, int64_t K, int64_t n_expert, int64_t n_used, int64_t T) {
    if (T * n_used < ROUTED_MIN_SLOTS || n_expert > 256 || K % QKK != 0 ||
        (type != MI355_Q4_K && type != MI355_Q5_K && type != MI355_Q6_K && type != MI355_IQ4_XS))
        return false;
    const row_layout L = make_row_layout(type, K);
    return layout_aligned(as, L) && (N * L.row_bytes) % 16 == 0;
}

// Between the two: the weight-streaming kernel, which reads every chosen expert's matrix once.  It pays from where the slots outnumber the
// experts they choose (on average E (1 - (1 - 1/E)^S) of E) by as much as it streams slower than the GEMV: 8 experts of 14336 x 4096,
// 8 / 12 / 24 slots: Q4_0 46 / 67 / 125 us with a GEMV per slot, 43 / 57 / 64 streamed; Q6_K 68 / 98 / 196 against 87 / 102 / 116.
// Up to 32 slots per expert it is ahead of the routed tile kernels (Q4_0, 32 / 64 / 256 / 512 slots: 214 / 208 / 215 / 245 us against
// 65 / 78 / 192 / 304; 16 experts of 2048 x 2048, 256 slots: 63 against 28; IQ4_XS 226 / 225 / 235 / 253 against 75 / 86 / 172 / 278); for the
// types whose routed kernel has 64-column tiles (routed, Q4_K and Q6_K) up to 16 (Q4_K, 32 / 64 / 128 / 256 slots: 147 / 146 / 149 / 154 us
// against 72 / 91 / 130 / 192; Q6_K 211 / 212 / 221 / 228 against 112 / 130 / 168 / 257).
// Those figures are for slots spread evenly.  Choices by Zipf's law: 8 experts of 14336 x 4096, 128 slots, Q4_K 134 us routed, 124 streamed; 256 of
// 512 x 2048, 8 per token, 1024 slots 89 / 51.  All tokens choosing the same two (eight) experts, where the routed kernel has full tiles: 8 experts, 64 /
// 128 slots Q4_K 56 / 58 routed, 47 / 68 streamed, Q4_0 148 / 154 against 44 / 67; 256 experts, 1024 slots Q4_K 40 / 50, Q6_K 43 / 73, Q4_0 100 / 52.
static bool use_skinny(int type, const void *as, int64_t K, int64_t n_expert, int64_t n_used, int64_t T, bool routed) {
    const int64_t S = T * n_used;
    const int64_t most = routed && (type == MI355_Q4_K || type == MI355_Q6_K) ? 16 : 32;
    if (!mi355_mul_mat_id_skinny_supported(type, as, K, n_expert, n_used, T) || S > most * n_expert) return false;
    const double chosen = (double)n_expert * (1.0 - pow(1.0 - 1.0 / (double)n_expert, (double)S));
    return (double)S >= (type == MI355_Q6_K ? 2.1 : 1.7) * chosen;
}

size_t mi355_mul_mat_id_ws_bytes(int64_t K, int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T) {
    const size_t act = (mi355_act_bytes(K, nb1 * T) + 255) & ~(size_t)255;   // the per-super-block format is the smaller one
    return act + mi355_mul_mat_id_q8k_route_bytes(n_expert, n_used, T);
}

int mi355_mul_mat_id(void *stream, int type, const void *as, const float *b, const int32_t *ids, int64_t ids_stride,
                     float *dst, int64_t N, int64_t K, int64_t n_expert, int64_t n_used, int64_t nb1, int64_t T,
                     void *ws, size_t ws_bytes) {
    MI355_REQUIRE(is_weight_type(type), "mul_mat_id: unsupported weight type %d", type);
    MI355_REQUIRE(N > 0 && K > 0 && n_expert > 0 && n_used > 0 && nb1 > 0 && T > 0, "mul_mat_id: bad shape");
    MI355_REQUIRE(K % type_block_elems(type) == 0, "mul_mat_id: K=%lld is not a multiple of the block size", (long long)K);
    MI355_REQUIRE(ids_stride >= n_used, "mul_mat_id: ids_stride < n_used");
    if (ws == nullptr || ws_bytes < mi355_mul_mat_id_ws_bytes(K, n_expert, n_used, nb1, T)) {
        set_error("mul_mat_id: workspace of %zu bytes, need %zu", ws_bytes, mi355_mul_mat_id_ws_bytes(K, n_expert, n_used, nb1, T));
        return MI355_ERR_WORKSPACE;
    }
    if (use_routed_tiles(type, as, N, K, n_expert, n_used, T)) {
        int rc = mi355_quantize_act_q8k(stream, b, ws, K, nb1 * T, K);
        if (rc != MI355_OK) return rc;
        if (use_skinny(type, as, K, n_expert, n_used, T, true)) return mi355_mul_mat_id_skinny_q8k(stream, type, as, ws, ids, ids_stride, dst, N, K, n_expert, n_used, nb1, T);
        const size_t act = (mi355_act_bytes(K, nb1 * T) + 255) & ~(size_t)255;
        return mi355_mul_mat_id_q8k(stream, type, as, ws, ids, ids_stride, dst, N, K, n_expert, n_used, nb1, T, (uint8_t *)ws + act,
                                    ws_bytes - act);
    }
    int rc = mi355_quantize_act(stream, b, ws, K, nb1 * T, K);
    if (rc != MI355_OK) return rc;
    if (use_skinny(type, as, K, n_expert, n_used, T, false)) return mi355_mul_mat_id_skinny(stream, type, as, ws, ids, ids_stride, dst, N, K, n_expert, n_used, nb1, T);
    if (T * n_used >= ROUTED_MIN_SLOTS && mi355_mul_mat_id_q_supported(type, as, N, K, n_expert)) {   // per-32-block types and the super-block types whose rows are no multiple of 16 bytes: the routed form of the per-block tile kernel
        const size_t act = (mi355_act_bytes(K, nb1 * T) + 255) & ~(size_t)255;
        return mi355_mul_mat_id_q(stream, type, as, ws, ids, ids_stride, dst, N, K, n_expert, n_used, nb1, T, (uint8_t *)ws + act, ws_bytes - act);
    }
    return mi355_mul_mat_id_vec(stream, type, as, ws, ids, ids_stride, dst, N, K, n_expert, n_used, nb1, T);
}

}  // extern "C"
