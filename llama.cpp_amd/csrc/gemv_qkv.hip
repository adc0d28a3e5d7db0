// The Q/K/V launches of one to four tokens: the three projections, ROPE and the stores to the KV cache, with the attention norm of a single token where asked for
// (gemv_body.hpp has the rows).
#include "gemv_body.hpp"

#include <math.h>

namespace mi355 {

// Q, K and V projections in one launch; finished rows are rotated and land in q (f32) or in the f16 KV cache
template <int NCOLS, bool LDSA>
__global__ void __launch_bounds__(256) k_gemv_qkv(gemv_batch b, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int K, gemv_rope rp) {
    const int g = blockIdx.x;
    int i = 0;
#pragma unroll
    for (int j = 1; j < 3; j++)
        if (g >= b.it[j].first_group) i = j;   // unused items start at INT_MAX
    const gemv_item &m = b.it[i];
    const int group = g - m.first_group;
#define MI355_BODY(TY) gemv_body<TY, NCOLS, 2, true, false, LDSA>(m, group, aq, ads, K, &rp, s_act_dyn);
    MI355_WEIGHT_TYPE_SWITCH(m.type, MI355_BODY)   // uniform over the group
#undef MI355_BODY
}

// ... with the RMS norm of the layer input computed by every group for itself (one activation row of at most 4096 elements).
//
// A launch of 13 MB takes 4.6 us in a chain of launches with the row already quantized; what it takes beyond that is the norm's dependent instructions and trips to memory that a wave
// makes one after the other.  So what the first requests need comes in arguments that are in registers when a wave starts (the first fourteen words), and where finished
// rows go and how they are rotated is read behind the requests for the weights: left to itself the compiler moves all those reads - the matrix's entry by its
// index, the rotation and the cell by what that holds - ahead of the branch over the types, and each waits for the one before it.  `late` is the index of the
// matrix, opaque from where those reads may begin.  Four waves and eight rows per group: the 768 groups of 8B shapes are three to every compute unit (eight waves are
// 384: two norms at a time on half of them, 7.2 us against 6.8; sixteen and 192 groups 9.2 against 8.4 in the previous form).
// 8B shapes, us in the chain: 8.4 with everything read first, 64-bit divisions for the head and four elements per lane and block piece; 6.8 now (a token 1608 -> 1553).
constexpr int QN_WAVES = 4;
struct qkv_rest {
    gemv_batch b;
    gemv_rope rp[1];
};
template <int TYPE, bool TABLE>
__device__ __forceinline__ void qkv_norm_body(const uint8_t *__restrict__ W, int64_t row0, int64_t last_row, const float *__restrict__ nx, const float *__restrict__ nw, int K,
                                              const qkv_rest &rest, int item) {
    typedef wq<TYPE> T;
    typedef late_chunk<TYPE> G;
    constexpr int STEPS = 64 / T::CHUNK;   // steps of 64 chunks in a row of 4096
    const int lane = threadIdx.x & 63;
    const row_layout L = make_row_layout(TYPE, K);
    const int nchunks = K / T::CHUNK;
    const uint8_t *rows[2];
#pragma unroll
    for (int r = 0; r < 2; r++) rows[r] = W + (row0 + r < last_row ? row0 + r : last_row) * L.row_bytes;   // rows past the end repeat the last one and are not stored
    __shared__ float s_norm[4];
    norm_row<QN_WAVES> row;
    row.request(nx, nw, K);
    __builtin_amdgcn_sched_barrier(0);
    typename G::raw w[STEPS][2];
#pragma unroll
    for (int p = 0; p < STEPS; p++)
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int c = p * 64 + lane;
            w[p][r] = G::load(rows[r], L, c < nchunks ? c : nchunks - 1);
        }
    __builtin_amdgcn_sched_barrier(0);
    int late = item;
    asm volatile("" : "+s"(late));
    const gemv_item &m = rest.b.it[late];
    const gemv_rope &R = rest.rp[late >> 2];   // (0)
    // one trip for what the rotation and the cell are looked up with, one for them, behind the weights (neither is waited for ahead of the sums; where a launch
    // has none of them some word of the row is read in their place)
    const int D = R.D, n_dims = R.n_dims, epi = m.epi;
    const int32_t *cells = R.cells;
    const float2 *table = R.table;
    const float eps = R.neps;
    float *dst = m.dst;
    const int64_t nb1 = m.nb1, nb2 = m.nb2;
    asm volatile("" ::"s"(D), "s"(n_dims), "s"(epi), "s"(cells), "s"(table), "s"(eps), "s"(dst), "s"(nb1), "s"(nb2));
    const u32 head = (u32)row0 / (u32)D;   // (2^31 rows of 1024 elements and more do not fit the memory)
    const int d = (int)((u32)row0 - head * (u32)D);
    const bool turned = (epi == EPI_ROPE || epi == EPI_ROPE_CACHE) && d < n_dims;
    int zero;   // an offset the compiler does not know to be the same in all lanes: it would wait for a uniform value at once, to keep it in a scalar register
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    float2 turn;
    if constexpr (TABLE) turn = (turned ? table + (d >> 1) : (const float2 *)nx)[zero];
    else if (turned) rope_coeffs(R, R.pos[0], d >> 1, turn.x, turn.y);
    const int cell = (epi == EPI_ROPE_CACHE || epi == EPI_CACHE ? cells : (const int32_t *)nx)[zero];
    __builtin_amdgcn_sched_barrier(0);
    row.finish(s_act_dyn, K, eps, s_norm);
    __syncthreads();
    float acc[2] = {0.0f, 0.0f};
#pragma unroll
    for (int p = 0; p < STEPS; p++) {
        const int c = p * 64 + lane;
        if (p * 64 >= nchunks) break;   // uniform
        const typename T::act A = T::load_a((const int8_t *)s_act_dyn, (const act_ds *)(s_act_dyn + K), c < nchunks ? c : nchunks - 1);
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const typename T::chunk now = G::decode(w[p][r], c);
            const float sum = T::accumulate(acc[r], now, A, T::dots(now, A));
            acc[r] = c < nchunks ? sum : acc[r];
        }
    }
    const float s0 = wave_sum_dpp(acc[0]), s1 = wave_sum_dpp(acc[1]);
    if (lane == 0 && row0 < last_row) {   // an even number of rows
        float y0 = s0, y1 = s1;
        if (turned) rope_apply(turn.x, turn.y, s0, s1, y0, y1);
        if (epi == EPI_ROPE || epi == EPI_STORE) {
            float *o = dst + row0;
            o[0] = y0;
            o[1] = y1;
        } else {
            _Float16 *o = (_Float16 *)((uint8_t *)dst + (int64_t)cell * nb1 + (int64_t)head * nb2) + d;
            o[0] = (_Float16)y0;
            o[1] = (_Float16)y1;
        }
    }
}
// first1, first2: first groups of the second and third matrix (`groups`, the number of all, where there is none); forms: five bits each for the types, from bit 15 three each for half
// the rows of a matrix's last group less one, from bit 24 K / 1024
template <bool TABLE>   // the rotations come from a table
__global__ void __launch_bounds__(64 * QN_WAVES) k_gemv_qkv_norm(const uint8_t *__restrict__ W0, const uint8_t *__restrict__ W1, const uint8_t *__restrict__ W2,
                                                                 const float *__restrict__ nx, const float *__restrict__ nw, int first1, int first2, int groups, u32 forms, qkv_rest rest) {
    const int g = blockIdx.x;
    const int item = g >= first2 ? 2 : g >= first1 ? 1 : 0;
    const uint8_t *W = item == 0 ? W0 : item == 1 ? W1 : W2;
    const int group = g - (item == 0 ? 0 : item == 1 ? first1 : first2);
    const int left = (item == 0 ? first1 : item == 1 ? first2 : groups) - g;   // groups of the matrix from this one on
    const int64_t row0 = ((int64_t)group * QN_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * 2;
    const int64_t last_row = (int64_t)(group + left - 1) * (2 * QN_WAVES) + ((forms >> (15 + 3 * item)) & 7) * 2 + 1;
    const int K = (int)(forms >> 24) << 10;
#define MI355_BODY(TY) qkv_norm_body<TY, TABLE>(W, row0, last_row, nx, nw, K, rest, item);
    MI355_WEIGHT_TYPE_SWITCH((int)((forms >> (5 * item)) & 31), MI355_BODY)   // uniform over the group
#undef MI355_BODY
}

// The same two launches with K and / or V going to a Q8_0 / Q4_0 cache (gemv_body_qc): 512 threads per group; the matrices with a
// quantized destination have groups of 32 rows, one cache block per group, the others groups of 16.  The host lists the groups
// of 32 rows first in the grid.
__device__ __forceinline__ int qkv_item_of(const gemv_batch &b, int g) {
    int i = 0, best = -1;
#pragma unroll
    for (int j = 0; j < 3; j++)
        if (g >= b.it[j].first_group && b.it[j].first_group > best) {   // unused items start at INT_MAX
            i = j;
            best = b.it[j].first_group;
        }
    return i;
}

template <int NCOLS>
__global__ void __launch_bounds__(512, (NCOLS == 1 ? 4 : 2)) k_gemv_qkv_qc(gemv_batch b, const int8_t *__restrict__ aq, const act_ds *__restrict__ ads, int K, gemv_rope rp) {
    const gemv_item &m = b.it[qkv_item_of(b, blockIdx.x)];
    const int group = blockIdx.x - m.first_group;
    if (m.epi >= EPI_ROPE_QCACHE) {   // uniform over the group
#define MI355_BODY(TY) gemv_body_qc<TY, NCOLS, false, true>(m, group, aq, ads, K, rp, nullptr);
        MI355_WEIGHT_TYPE_SWITCH(m.type, MI355_BODY)
#undef MI355_BODY
    } else {
#define MI355_BODY(TY) gemv_body_qc<TY, NCOLS, false, false>(m, group, aq, ads, K, rp, nullptr);
        MI355_WEIGHT_TYPE_SWITCH(m.type, MI355_BODY)
#undef MI355_BODY
    }
}

__global__ void __launch_bounds__(512, 4) k_gemv_qkv_norm_qc(gemv_batch b, int K, gemv_rope rp) {
    const gemv_item &m = b.it[qkv_item_of(b, blockIdx.x)];
    const int group = blockIdx.x - m.first_group;
    if (m.epi >= EPI_ROPE_QCACHE) {
#define MI355_BODY(TY) gemv_body_qc<TY, 1, true, true>(m, group, nullptr, nullptr, K, rp, s_act_dyn);
        MI355_WEIGHT_TYPE_SWITCH(m.type, MI355_BODY)
#undef MI355_BODY
    } else {
#define MI355_BODY(TY) gemv_body_qc<TY, 1, true, false>(m, group, nullptr, nullptr, K, rp, s_act_dyn);
        MI355_WEIGHT_TYPE_SWITCH(m.type, MI355_BODY)
#undef MI355_BODY
    }
}

}  // namespace mi355

using namespace mi355;

extern "C" {

// nx != null: one activation row that every group normalises and quantizes for itself (act is not read)
static int vec_q_rope_impl(void *stream, int n_mats, const mi355_gemv_rope_mat *mats, const void *act, int64_t K, int64_t B,
                             const mi355_rope_desc *rope, const float *nx, const float *nw, float neps, const void *table = nullptr) {
    MI355_REQUIRE(n_mats >= 1 && n_mats <= 3 && mats != nullptr && rope != nullptr, "mul_mat_vec_q_rope: 1..3 matrices per launch");
    MI355_REQUIRE(B >= 1 && B <= 4, "mul_mat_vec_q_rope: batch %lld outside 1..4", (long long)B);
    const int64_t D = rope->head_dim;
    const int n_dims = rope->n_dims;
    MI355_REQUIRE(D > 0 && D % 2 == 0 && n_dims > 0 && n_dims <= D && n_dims % 2 == 0, "mul_mat_vec_q_rope: bad head geometry");
    MI355_REQUIRE(rope->mode == 0, "mul_mat_vec_q_rope: only the adjacent-pair rope mode is fused (mode %d)", rope->mode);
    MI355_REQUIRE(nx != nullptr || ((uintptr_t)act & 15) == 0, "mul_mat_vec_q_rope: activation workspace is not 16-byte aligned");
    MI355_REQUIRE(nx == nullptr || (B == 1 && K <= 4096 && K % 1024 == 0 && ((uintptr_t)nx & 15) == 0 && ((uintptr_t)nw & 15) == 0),
                  "rms_norm_qkv_rope_store: one row of K <= 4096 (a multiple of 1024), 16-byte aligned x and weights");
    gemv_batch b;
    b.n = n_mats;
    int64_t groups = 0;
    bool needs_pos = false, needs_cells = false, any_qc = false;
    const int64_t group_rows = nx ? 2 * QN_WAVES : 8;
    for (int i = 0; i < n_mats; i++) any_qc = any_qc || mats[i].epilogue == MI355_EPI_ROPE_QCACHE || mats[i].epilogue == MI355_EPI_QCACHE;
    // groups of 32 rows (quantized-cache epilogues) first in the grid, then the groups of 8: pass 0 places the former
    for (int pass = 0; pass < 2; pass++) {
        for (int i = 0; i < 4; i++) {
            const mi355_gemv_rope_mat &m = mats[i < n_mats ? i : 0];
            const bool qc = m.epilogue == MI355_EPI_ROPE_QCACHE || m.epilogue == MI355_EPI_QCACHE;
            if (i < n_mats && qc != (pass == 0)) continue;
            if (i >= n_mats && pass == 0) continue;
            if (i < n_mats) {
                int rc = check_gemv_args("mul_mat_vec_q_rope", m.type, m.W, m.N, K, m.N);
                if (rc != MI355_OK) return rc;
                MI355_REQUIRE(m.epilogue >= MI355_EPI_STORE && m.epilogue <= MI355_EPI_QCACHE && m.dst != nullptr && m.N % 2 == 0,
                              "mul_mat_vec_q_rope: bad epilogue %d, missing destination or odd row count", m.epilogue);
                if (m.epilogue == MI355_EPI_STORE || m.epilogue == MI355_EPI_ROPE)
                    MI355_REQUIRE(m.dst_stride >= m.N, "mul_mat_vec_q_rope: dst_stride < N");
                else if (qc)
                    MI355_REQUIRE(((uintptr_t)m.dst & 1) == 0 && (m.dst_stride == MI355_Q8_0 || m.dst_stride == MI355_Q4_0) && m.nb1 >= 0 && m.nb2 >= 0 &&
                                      m.N % 32 == 0,
                                  "mul_mat_vec_q_rope: a quantized cache takes whole Q8_0 / Q4_0 blocks (N a multiple of 32)");
                else
                    MI355_REQUIRE(((uintptr_t)m.dst & 1) == 0 && m.nb1 % 2 == 0 && m.nb2 % 2 == 0, "mul_mat_vec_q_rope: misaligned f16 destination");
                if (m.epilogue != MI355_EPI_STORE) MI355_REQUIRE(m.N % D == 0, "mul_mat_vec_q_rope: N=%lld is not a whole number of heads", (long long)m.N);
                needs_pos = needs_pos || m.epilogue == MI355_EPI_ROPE || m.epilogue == MI355_EPI_ROPE_CACHE || m.epilogue == MI355_EPI_ROPE_QCACHE;
                needs_cells = needs_cells || m.epilogue == MI355_EPI_ROPE_CACHE || m.epilogue == MI355_EPI_CACHE || qc;
            }
            b.it[i].W = (const uint8_t *)m.W;
            b.it[i].residual = nullptr;
            b.it[i].N = m.N;
            b.it[i].type = m.type;
            b.it[i].dst = (float *)m.dst;
            b.it[i].dst_stride = m.dst_stride;
            b.it[i].nb1 = m.nb1;
            b.it[i].nb2 = m.nb2;
            b.it[i].ctype = qc ? (int)m.dst_stride : 0;
            // the kernel's epilogue codes: plain rows take the rope path with no rotation applied to them
            b.it[i].epi = m.epilogue == MI355_EPI_STORE        ? EPI_STORE
                          : m.epilogue == MI355_EPI_ROPE       ? EPI_ROPE
                          : m.epilogue == MI355_EPI_ROPE_CACHE ? EPI_ROPE_CACHE
                          : m.epilogue == MI355_EPI_CACHE      ? EPI_CACHE
                          : m.epilogue == MI355_EPI_ROPE_QCACHE ? EPI_ROPE_QCACHE
                                                               : EPI_QCACHE;
            b.it[i].first_group = i < n_mats ? (int)groups : 0x7fffffff;
            if (i < n_mats) groups += any_qc ? (qc ? m.N / 32 : (m.N + 15) / 16) : (m.N + group_rows - 1) / group_rows;   // 8 waves x 4 or 2 rows; without quantized stores 4 or 8 waves x 2 rows
        }
    }
    MI355_REQUIRE(table == nullptr || (nx != nullptr && !any_qc), "mul_mat_vec_q_rope: only the launch with the norm and f16 destinations reads a table");
    MI355_REQUIRE(!needs_pos || rope->pos != nullptr || table != nullptr, "mul_mat_vec_q_rope: rope positions missing");
    MI355_REQUIRE(!needs_cells || rope->cells != nullptr, "mul_mat_vec_q_rope: cache cells missing");
    MI355_REQUIRE(groups < 0x7fffffff, "mul_mat_vec_q_rope: too many rows for one launch");
    gemv_rope rp;
    rp.pos = needs_pos ? rope->pos : nullptr; rp.cells = needs_cells ? rope->cells : nullptr; rp.ff = rope->freq_factors;
    rp.D = (int)D; rp.n_dims = n_dims;
    rp.table = (const float2 *)table;
    rp.theta_scale = rp.freq_scale = rp.ext_factor = rp.attn_factor = rp.corr0 = rp.corr1 = 0.0f;
    if (!table) {
        rp.theta_scale = powf(rope->freq_base, -2.0f / n_dims);
        rp.freq_scale = rope->freq_scale; rp.ext_factor = rope->ext_factor; rp.attn_factor = rope->attn_factor;
        const float pi = 3.14159265358979323846f;   // ggml_rope_yarn_corr_dims, ggml/src/ggml.c:3695-3707
        const float c0 = floorf(n_dims * logf(rope->n_ctx_orig / (rope->beta_fast * 2 * pi)) / (2 * logf(rope->freq_base)));
        const float c1 = ceilf(n_dims * logf(rope->n_ctx_orig / (rope->beta_slow * 2 * pi)) / (2 * logf(rope->freq_base)));
        rp.corr0 = c0 > 0 ? c0 : 0;
        rp.corr1 = c1 < n_dims - 1 ? c1 : (float)(n_dims - 1);
    }
    hipStream_t s = (hipStream_t)stream;
    const int8_t *aq = (const int8_t *)act;
    const act_ds *ads = (const act_ds *)(aq + B * K);
    const size_t lds = act_lds_bytes((int)B, K, groups);
    if (nx != nullptr) {
        rp.nx = nx; rp.nw = nw; rp.neps = neps;
        if (any_qc) {
            MI355_LAUNCH(k_gemv_qkv_norm_qc, dim3((unsigned)groups), dim3(512), (size_t)K + K / 4, s, b, (int)K, rp);
            return launch_status("k_gemv_qkv_norm_qc");
        }
        u32 forms = 0;
        for (int i = 0; i < n_mats; i++) forms |= (u32)b.it[i].type << (5 * i) | (u32)((b.it[i].N / 2 - 1) % QN_WAVES) << (15 + 3 * i);
        forms |= (u32)(K / 1024) << 24;
        const qkv_rest rest = {b, {rp}};
        const int first1 = n_mats > 1 ? b.it[1].first_group : (int)groups, first2 = n_mats > 2 ? b.it[2].first_group : (int)groups;
#define MI355_QN_ARGS dim3((unsigned)groups), dim3(64 * QN_WAVES), (size_t)K + K / 4, s, b.it[0].W, b.it[1].W, b.it[2].W, nx, nw, first1, first2, (int)groups, forms, rest
        if (table) MI355_LAUNCH(k_gemv_qkv_norm<true>, MI355_QN_ARGS);
        else MI355_LAUNCH(k_gemv_qkv_norm<false>, MI355_QN_ARGS);
#undef MI355_QN_ARGS
        return launch_status("k_gemv_qkv_norm");
    }
    rp.nx = rp.nw = nullptr; rp.neps = 0.0f;
    if (any_qc) {   // every wave reads the activation from memory (L2): these launches have too few groups for the copy in LDS to pay
        switch (B) {
            case 1: MI355_LAUNCH((k_gemv_qkv_qc<1>), dim3((unsigned)groups), dim3(512), 0, s, b, aq, ads, (int)K, rp); break;
            case 2: MI355_LAUNCH((k_gemv_qkv_qc<2>), dim3((unsigned)groups), dim3(512), 0, s, b, aq, ads, (int)K, rp); break;
            case 3: MI355_LAUNCH((k_gemv_qkv_qc<3>), dim3((unsigned)groups), dim3(512), 0, s, b, aq, ads, (int)K, rp); break;
            default: MI355_LAUNCH((k_gemv_qkv_qc<4>), dim3((unsigned)groups), dim3(512), 0, s, b, aq, ads, (int)K, rp); break;
        }
        return launch_status("k_gemv_qkv_qc");
    }
    switch (B) {
        case 1:
            if (lds) MI355_LAUNCH((k_gemv_qkv<1, true>), dim3((unsigned)groups), dim3(256), lds, s, b, aq, ads, (int)K, rp);
            else MI355_LAUNCH((k_gemv_qkv<1, false>), dim3((unsigned)groups), dim3(256), 0, s, b, aq, ads, (int)K, rp);
            break;
        case 2:
            if (lds) MI355_LAUNCH((k_gemv_qkv<2, true>), dim3((unsigned)groups), dim3(256), lds, s, b, aq, ads, (int)K, rp);
            else MI355_LAUNCH((k_gemv_qkv<2, false>), dim3((unsigned)groups), dim3(256), 0, s, b, aq, ads, (int)K, rp);
            break;
        case 3:
            if (lds) MI355_LAUNCH((k_gemv_qkv<3, true>), dim3((unsigned)groups), dim3(256), lds, s, b, aq, ads, (int)K, rp);
            else MI355_LAUNCH((k_gemv_qkv<3, false>), dim3((unsigned)groups), dim3(256), 0, s, b, aq, ads, (int)K, rp);
            break;
        default:
            if (lds) MI355_LAUNCH((k_gemv_qkv<4, true>), dim3((unsigned)groups), dim3(256), lds, s, b, aq, ads, (int)K, rp);
            else MI355_LAUNCH((k_gemv_qkv<4, false>), dim3((unsigned)groups), dim3(256), 0, s, b, aq, ads, (int)K, rp);
            break;
    }
    return launch_status("k_gemv_qkv");
}

int mi355_mul_mat_vec_q_rope(void *stream, int n_mats, const mi355_gemv_rope_mat *mats, const void *act, int64_t K, int64_t B,
                             const mi355_rope_desc *rope) {
    return vec_q_rope_impl(stream, n_mats, mats, act, K, B, rope, nullptr, nullptr, 0.0f);
}

int mi355_rms_norm_mul_mat_vec_q_rope(void *stream, const float *x, const float *norm_w, float eps, int n_mats, const mi355_gemv_rope_mat *mats,
                                      int64_t K, const mi355_rope_desc *rope) {
    MI355_REQUIRE(x != nullptr && norm_w != nullptr, "rms_norm_mul_mat_vec_q_rope: missing operands");
    return vec_q_rope_impl(stream, n_mats, mats, nullptr, K, 1, rope, x, norm_w, eps);
}

int mi355_rms_norm_qkv_rope_store(void *stream, const float *x, const float *norm_w, float eps, int type_q, const void *wq, int type_k,
                                  const void *wk, int type_v, const void *wv, float *q, void *kcache, void *vcache, const int32_t *pos,
                                  const int32_t *cells, const float *freq_factors, int64_t K, int64_t H, int64_t HK, int64_t D, size_t k_nb1,
                                  size_t k_nb2, size_t v_nb1, size_t v_nb2, int n_dims, int mode, int n_ctx_orig, float freq_base,
                                  float freq_scale, float ext_factor, float attn_factor, float beta_fast, float beta_slow) {
    MI355_REQUIRE(H > 0 && HK > 0 && D > 0 && x != nullptr && norm_w != nullptr, "rms_norm_qkv_rope_store: bad head geometry or missing operands");
    mi355_gemv_rope_mat m[3];
    m[0] = mi355_gemv_rope_mat{type_q, wq, H * D, MI355_EPI_ROPE, q, H * D, 0, 0};
    m[1] = mi355_gemv_rope_mat{type_k, wk, HK * D, MI355_EPI_ROPE_CACHE, kcache, 0, (int64_t)k_nb1, (int64_t)k_nb2};
    m[2] = mi355_gemv_rope_mat{type_v, wv, HK * D, MI355_EPI_CACHE, vcache, 0, (int64_t)v_nb1, (int64_t)v_nb2};
    mi355_rope_desc r = {pos, cells, freq_factors, D, n_dims, mode, n_ctx_orig, freq_base, freq_scale, ext_factor, attn_factor, beta_fast, beta_slow};
    return vec_q_rope_impl(stream, 3, m, nullptr, K, 1, &r, x, norm_w, eps);
}

int mi355_rms_norm_qkv_rope_table_store(void *stream, const float *x, const float *norm_w, float eps, int type_q, const void *wq, int type_k, const void *wk,
                                        int type_v, const void *wv, float *q, void *kcache, void *vcache, const void *table, const int32_t *cells, int64_t K,
                                        int64_t H, int64_t HK, int64_t D, size_t k_nb1, size_t k_nb2, size_t v_nb1, size_t v_nb2, int n_dims) {
    MI355_REQUIRE(H > 0 && HK > 0 && D > 0 && x != nullptr && norm_w != nullptr, "rms_norm_qkv_rope_table_store: bad head geometry or missing operands");
    MI355_REQUIRE(table != nullptr && ((uintptr_t)table & 7) == 0, "rms_norm_qkv_rope_table_store: the table is missing or not 8-byte aligned");
    mi355_gemv_rope_mat m[3];
    m[0] = mi355_gemv_rope_mat{type_q, wq, H * D, MI355_EPI_ROPE, q, H * D, 0, 0};
    m[1] = mi355_gemv_rope_mat{type_k, wk, HK * D, MI355_EPI_ROPE_CACHE, kcache, 0, (int64_t)k_nb1, (int64_t)k_nb2};
    m[2] = mi355_gemv_rope_mat{type_v, wv, HK * D, MI355_EPI_CACHE, vcache, 0, (int64_t)v_nb1, (int64_t)v_nb2};
    mi355_rope_desc r = {nullptr, cells, nullptr, D, n_dims, 0, 0, 1.0f, 1.0f, 0.0f, 1.0f, 1.0f, 1.0f};
    return vec_q_rope_impl(stream, 3, m, nullptr, K, 1, &r, x, norm_w, eps, table);
}

int mi355_qkv_rope_store(void *stream, int type_q, const void *wq, int type_k, const void *wk, int type_v, const void *wv, const void *act,
                         float *q, void *kcache, void *vcache, const int32_t *pos, const int32_t *cells, const float *freq_factors,
                         int64_t K, int64_t B, int64_t H, int64_t HK, int64_t D, size_t k_nb1, size_t k_nb2, size_t v_nb1, size_t v_nb2,
                         int n_dims, int mode, int n_ctx_orig, float freq_base, float freq_scale, float ext_factor, float attn_factor,
                         float beta_fast, float beta_slow) {
    MI355_REQUIRE(H > 0 && HK > 0 && D > 0, "qkv_rope_store: bad head geometry");
    mi355_gemv_rope_mat m[3];
    m[0] = mi355_gemv_rope_mat{type_q, wq, H * D, MI355_EPI_ROPE, q, H * D, 0, 0};
    m[1] = mi355_gemv_rope_mat{type_k, wk, HK * D, MI355_EPI_ROPE_CACHE, kcache, 0, (int64_t)k_nb1, (int64_t)k_nb2};
    m[2] = mi355_gemv_rope_mat{type_v, wv, HK * D, MI355_EPI_CACHE, vcache, 0, (int64_t)v_nb1, (int64_t)v_nb2};
    mi355_rope_desc r = {pos, cells, freq_factors, D, n_dims, mode, n_ctx_orig, freq_base, freq_scale, ext_factor, attn_factor, beta_fast, beta_slow};
    return mi355_mul_mat_vec_q_rope(stream, 3, m, act, K, B, &r);
}

}  // extern "C"
