// Dispatch of the 4x4-MFMA paged decode kernel (ssq_decode_paged_q4.h) over its instantiation units.
#include "ssq_decode_paged_q4.h"

// Shapes this kernel serves (the caller has checked the layout -- 16-token pages, or contiguous rows
// at head_dim 128 with 128-dim values --, bf16/f16 V, alignment, code widths 0/4/6/8, and that masks
// and passthrough blocks (at most 16 dims) come with byte codes): head_dim 64 or 128, block_dim 1, 2,
// 4 or 8 with at most 64 blocks, value_dim 64 or 128, at most 256 codewords.
bool ssq_decode_q4_shape(const ssq_decode_args* a) {
    if (a->head_dim != 64 && a->head_dim != 128) return false;
    const int bd = a->block_dim;
    if (bd != 1 && bd != 2 && bd != 4 && bd != 8) return false;
    if (a->head_dim / bd > 64) return false;
    if (a->value_dim != 64 && a->value_dim != 128) return false;
    return a->n_centroids >= 1 && a->n_centroids <= kNC;
}

// LDS bytes for rg query rows per group and split_len tokens per split
size_t ssq_decode_q4_smem(const ssq_decode_args* a, int rg, int split_len) {
    return q4_smem(*a, 4 * ((rg + 3) / 4), split_len, SSQ_Q4_WAVES);
}

// whether the problem's instantiation has a length-balanced form (passthrough values as vectors)
bool ssq_decode_q4_has_cut(const ssq_decode_args* a, int rows) {
    return q4_cut(a->head_dim, (rows + 3) / 4, a->layout == SSQ_CONTIGUOUS, a->mask != nullptr, 0);
}
// LDS bytes of the length-balanced form with `pages` block-table slots
size_t ssq_decode_q4_cut_smem(const ssq_decode_args* a, int rg, int pages) {
    return q4_cut_smem(*a, 4 * ((rg + 3) / 4), pages, SSQ_Q4_WAVES);
}

// Combines the partials that the length-balanced decode left for sequences spanning several shares: one
// wave per query row, one lane per share for the (m, l) pairs; rows of sequences inside one share are
// already written.
__global__ __launch_bounds__(256) void k_merge_cut(const SsqPagedParams p) {
    const ssq_decode_args& a = p.a;
    const int lane = threadIdx.x & 63;
    const int rid = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (rid >= a.batch * a.num_q_heads * a.q_len) return;  // whole waves
    const int qi = rid % a.q_len;
    const int h = (rid / a.q_len) % a.num_q_heads;
    const int b = rid / (a.q_len * a.num_q_heads);
    const int kv = h / p.G, r = (h - kv * p.G) * a.q_len + qi;  // the row within its (sequence, KV head)
    const int Dv = a.value_dim;
    SsqCut ct;
    ct.init(a, lane, p.cut_wg, p.cut_seq, p.cut_min);
    if (ct.whole) return;
    int s, T;
    ct.locate(a, lane, b, p.cut_seq, s, T);
    const int e = s + T + p.cut_seq;
    const int w0 = s / ct.share, w1 = (e - 1) / ct.share;
    if (w0 == w1) return;
    float M = -INFINITY, L = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};  // dims lane + 64 k: value_dim <= 256
    for (int c0 = w0; c0 <= w1; c0 += 64) {
        const int w = c0 + lane, lo = w * ct.share;
        const bool in = w <= w1 && SsqCut::token(max(lo, s) - s, p.cut_seq, T) <
                                       SsqCut::token(min(lo + ct.share, e) - s, p.cut_seq, T);
        const int at = (2 * (w * a.num_kv_heads + kv) + (s <= lo ? 0 : 1)) * p.rows + r;
        const float m = in ? p.ws_m[at] : -INFINITY;
        const float l = in ? p.ws_l[at] : 0.f;
        const float Mc = fmaxf(M, ssq_wave_max(m));
        const float f = M == -INFINITY ? 0.f : __expf(M - Mc);
        const float wt = m == -INFINITY ? 0.f : __expf(m - Mc);
        L = L * f + ssq_wave_sum(l * wt);
        M = Mc;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] *= f;
        // every share's values, also at weight 0: 0 times an infinite or NaN value is NaN, as in one pass
        const uint64_t live = __builtin_amdgcn_ballot_w64(in);
        for (uint64_t t = live; t; t &= t - 1) {
            const int i = __builtin_ctzll(t);
            const float wi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wt), i));
            const size_t row = (size_t)__builtin_amdgcn_readlane(at, i) * Dv;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (64 * k < Dv) o[k] += p.ws_o[row + min(64 * k + lane, Dv - 1)] * wi;
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int dv = 64 * k + lane;
        if (dv < Dv)
            ssq_store_elem(a.out, a.v_dtype, (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)qi * a.o_sl + dv, o[k] / L);
    }
    if (a.lse && lane == 0) a.lse[rid] = M + logf(L);
}

int ssq_decode_q4_merge_cut(const SsqPagedParams& mp, hipStream_t st) {
    const int rows = mp.a.batch * mp.a.num_q_heads * mp.a.q_len;
    hipLaunchKernelGGL(k_merge_cut, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, mp);
    return ssq_check_hip(hipGetLastError(), "k_merge_cut launch");
}

// Launches the 4x4-MFMA kernel for a planned problem (grid: batch*KV heads, splits, row groups);
// mp.rg rows per group (<= 16).  The caller launches the split merge.
int ssq_decode_q4_launch(const SsqPagedParams& mp, const dim3& grid, hipStream_t st) {
    const int R4 = (mp.rg + 3) / 4;
    const int DT = mp.a.value_dim / 16;
    const size_t smem = 0;  // launch_q4 sizes the LDS for its wave count
    const bool bf = mp.a.v_dtype == SSQ_BF16;
    const bool packed = mp.a.code_bits == 4 || mp.a.code_bits == 6;
    const bool mixed = mp.a.mask != nullptr || mp.a.heavy_mask[0] != 0;  // byte codes (the plan checks)
    if (mixed && (packed || mp.a.heavy_mask[1] != 0))
        return ssq_fail(SSQ_ERR_UNSUPPORTED, "4x4-MFMA decode: masks and passthrough need byte codes, blocks < 64");
    if (mp.a.layout == SSQ_CONTIGUOUS) {  // contiguous rows: head_dim 128, 128-dim values
        if (mp.a.head_dim != 128) return ssq_fail(SSQ_ERR_UNSUPPORTED, "4x4-MFMA decode: contiguous rows at head_dim %d",
                                                  mp.a.head_dim);
        if (mixed) return bf ? ssq_q4ct_128_bf16_mixed(mp, R4, DT, grid, smem, st) : ssq_q4ct_128_f16_mixed(mp, R4, DT, grid, smem, st);
        if (bf) return packed ? ssq_q4ct_128_bf16_packed(mp, R4, DT, grid, smem, st) : ssq_q4ct_128_bf16_bytes(mp, R4, DT, grid, smem, st);
        return packed ? ssq_q4ct_128_f16_packed(mp, R4, DT, grid, smem, st) : ssq_q4ct_128_f16_bytes(mp, R4, DT, grid, smem, st);
    }
    if (mixed) {
        if (mp.a.head_dim == 64)
            return bf ? ssq_q4_64_bf16_mixed(mp, R4, DT, grid, smem, st) : ssq_q4_64_f16_mixed(mp, R4, DT, grid, smem, st);
        return bf ? ssq_q4_128_bf16_mixed(mp, R4, DT, grid, smem, st) : ssq_q4_128_f16_mixed(mp, R4, DT, grid, smem, st);
    }
    if (mp.a.head_dim == 64) {
        if (bf) return packed ? ssq_q4_64_bf16_packed(mp, R4, DT, grid, smem, st) : ssq_q4_64_bf16_bytes(mp, R4, DT, grid, smem, st);
        return packed ? ssq_q4_64_f16_packed(mp, R4, DT, grid, smem, st) : ssq_q4_64_f16_bytes(mp, R4, DT, grid, smem, st);
    }
    if (bf) return packed ? ssq_q4_128_bf16_packed(mp, R4, DT, grid, smem, st) : ssq_q4_128_bf16_bytes(mp, R4, DT, grid, smem, st);
    return packed ? ssq_q4_128_f16_packed(mp, R4, DT, grid, smem, st) : ssq_q4_128_f16_bytes(mp, R4, DT, grid, smem, st);
}
