// VQ-key decode for 16-bit codes (4,096 codewords of dim 4 at 3 bits/dim, 1,024 of dim 2 at 5, ...)
// over long contexts: the codebook staged in LDS one block at a time for a super-tile of tokens.
//
// The per-token path (k_decode_generic, 16-bit-code variants) gathers each token's codeword of each
// block from the codebook in memory: one random 16-byte read per (token, block), an L2 line each,
// and the gathers bound it.  Here a workgroup takes a super-tile of up to 4,096 tokens of one
// (batch, KV head) and walks the blocks in order: block blk's codebook (nc * bd floats, at most
// 64 KiB) is copied into LDS once, every token's codeword of that block is read from there, and
// its scores (one per query row, at most 4 rows per workgroup) are accumulated in registers.
// Block blk + 1's codebook goes into the other half of a double buffer while blk is computed
// (direct global-to-LDS loads issued before blk's arithmetic), so one workgroup barrier per
// block separates them.
//
// Scores and P.V on 4x4 matrix-core blocks, in fp32.  v_mfma_f32_4x4x1_16b_f32 with the A operand
// broadcast from one block (cbsz, abid) multiplies 4 rows with every lane's own value: 4 rows x 64
// values per 8 matrix-core cycles, twice the VALU's rate, and the VALU is left to addresses and adds.
//   scores: A = the query rows' dim, B = the lane's token's codeword element; a block's chain starts
//           from zero (the LUT entry's FMA chain) and is added to the token's scores in block order,
//           so the raw scores equal the per-token path's bit for bit.
//   P.V:    A = 16 tokens' probabilities (fp32, from LDS), B = the lane's value element: 2 dims of a
//           token per lane on contiguous rows, 1 dim of 8 tokens on pages.  A lane keeps 2 x 4
//           accumulators, which leaves 16 waves' 128 registers room for the code rows.  At 64 value dims
//           a batch takes two 16-token runs, so that as many bytes are in flight as at 128 (16 x 8 x 8,192
//           tokens, 16 blocks of dim 4, 512 codewords, 4 query rows: pages 81 -> 58 us, rows 60 -> 53).
//
// Then per super-tile: mask, optional raw-score store, the softmax update (the super-tile's row
// maximum), P.V over the super-tile's V rows, and at the end of the split the normalised output +
// lse, or (m, l, o) partials for k_merge -- the same outputs and workspace layout as k_decode_generic
// (sunshape/vllm_attn_backend.py:216-253; scores sunshape/triton_kernels.py:174-196, LUT entries
// :381-408).
//
// 1024 threads (16 waves), one workgroup per CU (the double buffer is 128 KiB at 4,096 codewords of
// dim 4).  4 tokens per thread where a split holds more than 2,048 tokens (a codebook copy per 4,096
// tokens), 2 below.  32 blocks' codes of each token stay in registers (16 where there are no more), so a
// 64-byte row is read once.
//
// What bounds it, at 32 sequences x 8 KV heads x 16,384 tokens, 4 query rows, 4,096 codewords of dim 4,
// 128 value dims (1.36 GB; 270 us at a copy's rate): 411 us, of which P.V 146 us (at 7.3 TB/s), the 32
// blocks 210 us (1.4 us per block of 4,096 tokens: a 64 KiB copy into LDS, 64 KiB of random 16-byte
// reads out of it and a barrier; 0.84 us at 512 codewords, where the copy is 8 KiB), the rest code rows.
// 512 threads of 8 tokens with FMA chains on the VALU and rows read 16 bytes at a time took 502 us;
// 1024 threads of 8 tokens, rows 16 bytes at a time, 437; 512 threads of 8 tokens with whole rows and a
// block's reads issued under the products of the block before, 505 (too few waves).  Super-tiles
// staggered over the sequences, so that one's P.V meets another's blocks, made an earlier form of this
// kernel slower, 395 -> 426 (a fifth pass costs more than the overlap gives).  Splits of 2,048 tokens:
// 92 -> 65 us, of 4,096: 136 -> 104.  At 128 value dims P.V takes 16 tokens per wave and batch: 32 are no
// faster, 64 on pages 10 to 25 % slower.
//
// Host-checked: 16-bit codes in 16-byte aligned rows of a multiple of 8
// blocks (at most 64), codewords of 2 or 4 dims in a 16-byte aligned codebook of at most 64 KiB per
// block, no passthrough blocks, bf16 or f16 values of 64 or 128 dims.
#include "ssq_decode_generic.h"

#include <type_traits>

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kWT = 1024;                // threads per workgroup
constexpr int kWWaves = kWT / SSQ_WAVE;  // 16

// tokens per thread per super-tile (the super-tile is kWT times that) for splits of split_len tokens
inline int wide_tpt(int split_len) { return split_len > 2 * kWT ? 4 : 2; }

// LDS layout, in floats: [stage / p / obuf | qp | red | pgl]
struct WideLds {
    size_t qp, red, pgl, total;
};
__host__ __device__ inline WideLds wide_lds(const ssq_decode_args& a, int RP, int tpt) {
    const size_t ncb = (size_t)a.n_centroids * a.block_dim;
    const size_t sup = (size_t)tpt * kWT;
    size_t r0 = 2 * ncb;                                              // double-buffered codebook stage
    if ((size_t)RP * sup > r0) r0 = (size_t)RP * sup;                 // the super-tile's p
    if ((size_t)kWWaves * RP * a.value_dim > r0) r0 = (size_t)kWWaves * RP * a.value_dim;  // epilogue
    WideLds l;
    l.qp = (r0 + 3) & ~(size_t)3;
    l.red = l.qp + (size_t)RP * a.head_dim;
    l.pgl = l.red + 2 * kWWaves * RP;
    l.total = l.pgl + sup / 8;
    return l;
}

// acc + a_row * b over 4x4 blocks: A from block J of each group of 2^CBSZ blocks
template <int CBSZ, int J>
__device__ __forceinline__ v4f mfma4(float a, float b, v4f acc) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc, CBSZ, J, 0);
}
template <int B, int E, typename F>
__device__ __forceinline__ void for_each_const(const F& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        for_each_const<B + 1, E>(f);
    }
}
template <int VT>
__device__ __forceinline__ float val_lo(uint32_t w) {
    return VT == SSQ_BF16 ? __uint_as_float(w << 16) : ssq_f16_to_f32(w & 0xFFFFu);
}
template <int VT>
__device__ __forceinline__ float val_hi(uint32_t w) {
    return VT == SSQ_BF16 ? __uint_as_float(w & 0xFFFF0000u) : ssq_f16_to_f32(w >> 16);
}

// One block's codebook (n4 16-byte pieces, at most kStagePieces * kWT) into an LDS stage half with direct
// global-to-LDS loads: wave w's u-th load puts its 64 lanes' pieces u * kWT + 64 w + lane at the
// wave's LDS base + 16 * lane (lanes past n4 are inactive).  Completion is waited for with vmcnt.
constexpr int kStagePieces = 4;
__device__ __forceinline__ void stage_block_lds(const float* src_blk, float* half, int n4, int tid) {
    const int wbase = tid & ~(SSQ_WAVE - 1);
#pragma unroll
    for (int u = 0; u < kStagePieces; ++u) {
        const int i = u * kWT + tid;
        if (i < n4)
            __builtin_amdgcn_global_load_lds(static_cast<const void*>(src_blk + (size_t)i * 4),
                                             (__attribute__((address_space(3))) void*)(half + (size_t)(u * kWT + wbase) * 4),
                                             16, 0, 0);
    }
}

// BD: the block dim, 2 or 4 (the plan's condition), fixed at compile time so that each token's
// codeword is one LDS read and its FMA chain carries no branches.  TPT: tokens per thread.  NP: 16-byte
// pieces of 8 blocks' codes held in registers, 4, or 2 up to 16 blocks.
template <int RP, bool PAGED, int VT, int BD, int TPT, int NP>
__global__ __launch_bounds__(kWT) void k_decode_wide(const SsqGenericParams p) {
    extern __shared__ __align__(16) float smem[];
    const ssq_decode_args& a = p.a;
    constexpr int kK = TPT;
    constexpr int kSup = kK * kWT;
    constexpr int kPieces = NP;
    const WideLds L = wide_lds(a, RP, TPT);
    const int tid = threadIdx.x;
    const int lane = tid & (SSQ_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / SSQ_WAVE);
    const int split = blockIdx.x;
    const int grp = blockIdx.y;
    const int bk = blockIdx.z;
    const int b = bk / a.num_kv_heads;
    const int kv = bk - b * a.num_kv_heads;
    const int nb = a.n_blocks, nc = a.n_centroids, D = a.head_dim, Dv = a.value_dim;
    const int r0 = grp * p.R;
    const int nr = min(p.R, p.rows - r0);
    const int T = PAGED ? min(a.seq_lens[b], a.seq_len) : a.seq_len;
    const int t_begin = split * p.split_len;
    const int t_end = min(T, t_begin + p.split_len);
    const int ncb = nc * BD;
    const int n4 = ncb / 4;  // float4s of one block's codebook: at most 4 per thread (host-checked)
    float* stage = smem;     // [2][ncb]
    float* pbuf = smem;      // [RP][kSup], after a super-tile's blocks
    float* qp = smem + L.qp;
    float* red = smem + L.red;
    int* pgl = reinterpret_cast<int*>(smem + L.pgl);

    // ---- scaled, permuted query rows (as k_decode_generic)
    const int64_t* perm = a.perm + (int64_t)kv * a.perm_sh;
    for (int e0 = 0; e0 < RP * D; e0 += 4 * kWT) {
        int64_t src[4];
        bool ok[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = e0 + k * kWT + tid;
            src[k] = perm[e < RP * D ? e % D : 0];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = e0 + k * kWT + tid;
            const int r = e / D;
            ok[k] = e < RP * D && r < nr;
            if (ok[k]) {
                const int row = r0 + r;
                const int g = row / a.q_len, qi = row - g * a.q_len;
                const int h = kv * p.G + g;
                src[k] += (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)qi * a.q_sl;
            }
        }
        float v[4];
        ssq_load_elems(a.q, a.q_dtype, src, v);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = e0 + k * kWT + tid;
            if (e < RP * D) qp[e] = !ok[k] ? 0.f : a.has_scale ? ssq_round_to(v[k] * a.scale, a.q_dtype) : v[k];
        }
    }

    const float* cent = a.cent + (int64_t)kv * a.cent_sh;
    const uint16_t* codes = reinterpret_cast<const uint16_t*>(a.codes);
    float m_run[RP], l_thr[RP];
#pragma unroll
    for (int r = 0; r < RP; ++r) { m_run[r] = -INFINITY; l_thr[r] = 0.f; }
    // P.V: acc[e] is rows 0..3 of one dim: contiguous rows 2 (lane % (Dv / 2)) + e, pages lane + 64 e
    v4f acc[2];
    acc[0] = acc[1] = (v4f){0.f, 0.f, 0.f, 0.f};
    // A operands: lane 4 j + i holds row i's value of dim (scores) or token (P.V) j
    const int arow = lane & 3, aj = lane >> 2;

    for (int T0 = t_begin; T0 < t_end; T0 += kSup) {
        if (PAGED) {  // the page of each 8-token chunk, for the P.V loads (page_size % 8 == 0)
            for (int c = tid; c < kSup / 8; c += kWT) {
                const int t = min(T0 + 8 * c, t_end - 1);
                pgl[c] = a.block_table[(int64_t)b * a.bt_sb + t / a.page_size];
            }
        }
        float ss[kK][RP];
#pragma unroll
        for (int k = 0; k < kK; ++k)
#pragma unroll
            for (int r = 0; r < RP; ++r) ss[k][r] = 0.f;

        // a thread's tokens are T0 + k * kWT + tid (past t_end: the last token's row, not used); w holds up
        // to 32 blocks' codes of each, read once: 8 blocks (16 bytes) at a time would fetch every 64-byte
        // row four times, and a super-tile of all workgroups' rows is larger than L2
        ssq_v4u w[kK][kPieces];
        auto load_rows = [&](int blk0) {
#pragma unroll
            for (int k = 0; k < kK; ++k) {
                const int t = min(T0 + k * kWT + tid, t_end - 1);
                int64_t row = (int64_t)kv * a.c_sh + blk0;
                if (PAGED) {
                    const int pg = t / a.page_size;
                    row += (int64_t)a.block_table[(int64_t)b * a.bt_sb + pg] * a.c_sb + (int64_t)(t - pg * a.page_size) * a.c_st;
                } else {
                    row += (int64_t)b * a.c_sb + (int64_t)t * a.c_st;
                }
#pragma unroll
                for (int i = 0; i < kPieces; ++i)
                    w[k][i] = *reinterpret_cast<const ssq_v4u*>(codes + row + min(8 * i, nb - 8 - blk0));
            }
        };
        load_rows(0);
        // block 0's codebook into stage half 0 (the previous super-tile's p reads are done: the
        // barrier that ended its P.V)
        stage_block_lds(cent, stage, n4, tid);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
#pragma unroll 1
        for (int b8 = 0; b8 < nb; b8 += 8) {
            constexpr int kQA = 8 * BD / 16;  // A registers of 8 blocks' dims
            float qa[kQA];
#pragma unroll
            for (int i = 0; i < kQA; ++i) qa[i] = arow < RP ? qp[min(arow, RP - 1) * D + b8 * BD + 16 * i + aj] : 0.f;
            for_each_const<0, 8>([&](auto kbc) {
                constexpr int kb = decltype(kbc)::value;
                const int blk = b8 + kb;
                uint32_t cw[kK];  // this block's codeword of each token
#pragma unroll
                for (int k = 0; k < kK; ++k) {
                    uint32_t pair = kb < 2 ? w[k][0].x : kb < 4 ? w[k][0].y : kb < 6 ? w[k][0].z : w[k][0].w;
                    __asm__ volatile("" : "+v"(pair));  // extracted in this block, not 8 blocks ahead
                    cw[k] = min((kb & 1) ? pair >> 16 : pair & 0xFFFFu, (uint32_t)(nc - 1));
                }
                if (kb == 7) {  // piece 0 is spent
                    if ((blk + 1) % (8 * kPieces) == 0) {
                        if (blk + 1 < nb) load_rows(blk + 1);  // in flight during this block
                    } else {
#pragma unroll
                        for (int k = 0; k < kK; ++k)
#pragma unroll
                            for (int i = 0; i + 1 < kPieces; ++i) w[k][i] = w[k][i + 1];
                    }
                }
                const float* cur = stage + (size_t)(kb & 1) * ncb;  // nb is a multiple of 8
                // the next block's codebook into the other half (last read in the previous block,
                // before its barrier), in flight during this block's arithmetic
                if (blk + 1 < nb)
                    stage_block_lds(cent + (int64_t)(blk + 1) * ncb, stage + (size_t)((kb + 1) & 1) * ncb, n4, tid);
#pragma unroll
                for (int k = 0; k < kK; ++k) {
                    float c[BD];
                    if constexpr (BD == 4) {
                        const float4 v4 = *reinterpret_cast<const float4*>(cur + (size_t)cw[k] * 4);
                        c[0] = v4.x; c[1] = v4.y; c[2] = v4.z; c[3] = v4.w;
                    } else {
                        const float2 v2 = *reinterpret_cast<const float2*>(cur + (size_t)cw[k] * 2);
                        c[0] = v2.x; c[1] = v2.y;
                    }
                    v4f e = {0.f, 0.f, 0.f, 0.f};
                    for_each_const<0, BD>([&](auto dc) {
                        constexpr int d = decltype(dc)::value, kd = kb * BD + d;
                        e = mfma4<4, (kd & 15)>(qa[kd >> 4], c[d], e);
                    });
#pragma unroll
                    for (int r = 0; r < RP; ++r) {
                        ss[k][r] += e[r];
                        __asm__ volatile("" : "+v"(ss[k][r]));  // added here (sinking the adds spills every e)
                    }
                }
                __builtin_amdgcn_s_waitcnt(0);  // the next half (and reloaded code pieces) has landed
                __syncthreads();
            });
        }

        // ---- mask, raw scores, softmax update
        float mx[RP];
#pragma unroll
        for (int r = 0; r < RP; ++r) mx[r] = -INFINITY;
#pragma unroll
        for (int k = 0; k < kK; ++k) {
            const int t = T0 + k * kWT + tid;
            const bool valid = t < t_end;
            if (valid && a.mask) {
                float mk[RP];
#pragma unroll
                for (int r = 0; r < RP; ++r) {
                    const int row = r0 + (r < nr ? r : 0);
                    const int g = row / a.q_len, qi = row - g * a.q_len;
                    const int h = kv * p.G + g;
                    mk[r] = a.mask[(int64_t)b * a.m_sb + (int64_t)h * a.m_sh + (int64_t)qi * a.m_sl + (int64_t)t * a.m_st];
                }
#pragma unroll
                for (int r = 0; r < RP; ++r)
                    if (r < nr) ss[k][r] += mk[r];
            }
            if (valid && a.scores) {
#pragma unroll
                for (int r = 0; r < RP; ++r) {
                    if (r < nr) {
                        const int row = r0 + r;
                        const int g = row / a.q_len, qi = row - g * a.q_len;
                        const int h = kv * p.G + g;
                        a.scores[(int64_t)b * a.s_sb + (int64_t)h * a.s_sh + (int64_t)qi * a.s_sl + t] = ss[k][r];
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < RP; ++r) mx[r] = fmaxf(mx[r], valid ? ss[k][r] : -INFINITY);
        }
#pragma unroll
        for (int r = 0; r < RP; ++r) {
            const float v = ssq_wave_max(mx[r]);
            if (lane == 0) red[wave * RP + r] = v;
        }
        __syncthreads();
        float alpha[RP];
#pragma unroll
        for (int r = 0; r < RP; ++r) {
            float tm = red[r];
#pragma unroll
            for (int w2 = 1; w2 < kWWaves; ++w2) tm = fmaxf(tm, red[w2 * RP + r]);
            const float mn = fmaxf(m_run[r], tm);
            alpha[r] = (mn == -INFINITY) ? 1.f : __expf(m_run[r] - mn);
            m_run[r] = mn;
            float lsum = 0.f;
#pragma unroll
            for (int k = 0; k < kK; ++k) {
                const int tt = k * kWT + tid;
                const float pr = (T0 + tt < t_end && mn != -INFINITY) ? __expf(ss[k][r] - mn) : 0.f;
                lsum += pr;
                pbuf[(size_t)r * kSup + tt] = pr;
            }
            l_thr[r] = l_thr[r] * alpha[r] + lsum;
        }
#pragma unroll
        for (int r = 0; r < RP; ++r) {
            acc[0][r] *= alpha[r];
            acc[1][r] *= alpha[r];
        }
        __syncthreads();

        // ---- P.V over the super-tile's nt tokens, 16 at a time per wave; a batch's loads are issued
        // before their arithmetic (clamped to the last token / chunk, whose p is then 0)
        const int nt = min(kSup, t_end - T0);
        const int groups = (nt + 15) >> 4;
        auto probs = [&](int g) {  // 16 tokens' A operand (p past the end is 0)
            return arow < RP ? pbuf[(size_t)min(arow, RP - 1) * kSup + g * 16 + aj] : 0.f;
        };
        if (!PAGED) {
            // a lane's 4 bytes are 2 dims: a wave's load is one token's row (128 dims) or two tokens'
            // (64 dims: the lanes' halves take tokens j and j + 8)
            const uint16_t* vb = reinterpret_cast<const uint16_t*>(a.v) + (int64_t)b * a.v_sb + (int64_t)kv * a.v_sh +
                                 (int64_t)T0 * a.v_st;
            if (Dv == 128) {
                for (int g = wave; g < groups; g += kWWaves) {
                    uint32_t raw[16];
#pragma unroll
                    for (int k = 0; k < 16; ++k)
                        raw[k] = __builtin_nontemporal_load(
                            reinterpret_cast<const uint32_t*>(vb + (int64_t)min(g * 16 + k, nt - 1) * a.v_st) + lane);
                    const float pa = probs(g);
                    __asm__ volatile("" ::: "memory");  // the batch's loads stay ahead of every use
                    if ((g + 1) * 16 > nt) {  // clamped slots: 0, not p = 0 times a value that may be infinite
#pragma unroll
                        for (int k = 0; k < 16; ++k) raw[k] = g * 16 + k < nt ? raw[k] : 0u;
                    }
                    for_each_const<0, 16>([&](auto kc) {
                        constexpr int k = decltype(kc)::value;
                        acc[0] = mfma4<4, k>(pa, val_lo<VT>(raw[k]), acc[0]);
                        acc[1] = mfma4<4, k>(pa, val_hi<VT>(raw[k]), acc[1]);
                    });
                }
            } else {
                const int hl = lane >> 5;
                for (int g0 = 2 * wave; g0 < groups; g0 += 2 * kWWaves) {  // two groups: as many loads as at 128 dims
                    uint32_t raw[16];
                    float pa[2];
#pragma unroll
                    for (int k = 0; k < 16; ++k)
                        raw[k] = __builtin_nontemporal_load(
                            reinterpret_cast<const uint32_t*>(
                                vb + (int64_t)min((g0 + (k >> 3)) * 16 + 8 * hl + (k & 7), nt - 1) * a.v_st) + (lane & 31));
                    pa[0] = probs(g0);
                    pa[1] = g0 + 1 < groups ? probs(g0 + 1) : 0.f;
                    __asm__ volatile("" ::: "memory");
                    if ((g0 + 2) * 16 > nt) {
#pragma unroll
                        for (int k = 0; k < 16; ++k)
                            raw[k] = (g0 + (k >> 3)) * 16 + 8 * hl + (k & 7) < nt ? raw[k] : 0u;
                    }
                    for_each_const<0, 16>([&](auto kc) {
                        constexpr int k = decltype(kc)::value;
                        acc[0] = mfma4<3, (k & 7)>(pa[k >> 3], val_lo<VT>(raw[k]), acc[0]);
                        acc[1] = mfma4<3, (k & 7)>(pa[k >> 3], val_hi<VT>(raw[k]), acc[1]);
                    });
                }
            }
        } else {
            // a lane's 16 bytes are 8 tokens of its dim; both halves of a 16-token run are loaded back to
            // back, so a run's line is fetched once, and two runs at a time: the run of both of the
            // lane's dims (128), or two runs of its dim (64; acc[1] then holds the second run's sums)
            const int nchunks = (nt + 7) >> 3;
            const int64_t vhead = (int64_t)kv * a.v_sh + (int64_t)lane * a.v_st;
            auto pages_pv = [&](auto two_runs) {
            constexpr bool two = decltype(two_runs)::value;
            constexpr int step = two ? 2 : 1;
            for (int g0 = wave * step; g0 < groups; g0 += kWWaves * step) {
                VRaw8<VT> raw[2][2];  // [dim or run][half]
                float pa[2];
                int64_t src[2][2];
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int c = min(2 * (g0 + (two ? e : 0)) + h, nchunks - 1);
                        const int t = T0 + 8 * c;
                        src[e][h] = (int64_t)pgl[c] * a.v_sb + vhead + (two ? 0 : 64 * e) * a.v_st +
                                    (t - (t / a.page_size) * a.page_size);
                    }
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int h = 0; h < 2; ++h) raw[e][h] = load_v8_raw<VT, true>(a.v, src[e][h]);
                pa[0] = probs(g0);
                pa[1] = !two ? pa[0] : g0 + 1 < groups ? probs(g0 + 1) : 0.f;
                __asm__ volatile("" ::: "memory");
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int g = g0 + (two ? e : 0);
                    float v[16];
                    float lo8[8], hi8[8];
                    unpack_v8<VT>(raw[e][0], lo8);
                    unpack_v8<VT>(raw[e][1], hi8);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        v[j] = lo8[j];
                        v[8 + j] = hi8[j];
                    }
                    if ((g + 1) * 16 > nt) {  // values of slots past the end are unwritten
#pragma unroll
                        for (int j = 0; j < 16; ++j) v[j] = g * 16 + j < nt ? v[j] : 0.f;
                    }
                    for_each_const<0, 16>([&](auto jc) {
                        constexpr int j = decltype(jc)::value;
                        acc[e] = mfma4<4, j>(pa[e], v[j], acc[e]);
                    });
                }
            }
            };
            if (Dv == 64) pages_pv(std::true_type{});
            else pages_pv(std::false_type{});
        }
        __syncthreads();  // p and pgl are read before the next super-tile's stage / pages
    }

    // ---- epilogue: l summed over threads, o over waves (and, 64 contiguous dims, over lane halves)
    float* red2 = red + kWWaves * RP;
#pragma unroll
    for (int r = 0; r < RP; ++r) {
        const float v = ssq_wave_sum(l_thr[r]);
        if (lane == 0) red2[wave * RP + r] = v;
    }
    float* obuf = smem;  // [waves][RP][Dv]
    if (!PAGED && Dv == 64) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int r = 0; r < RP; ++r) acc[e][r] += __shfl_xor(acc[e][r], 32, SSQ_WAVE);
    }
    if (PAGED && Dv == 64) acc[0] += acc[1];
    const int d_lane = PAGED ? lane : 2 * (Dv == 64 ? lane & 31 : lane), d_step = PAGED ? 64 : 1;
#pragma unroll
    for (int e = 0; e < 2; ++e)
        if (!PAGED || e < (Dv >> 6)) {
#pragma unroll
            for (int r = 0; r < RP; ++r) obuf[((size_t)wave * RP + r) * Dv + d_lane + e * d_step] = acc[e][r];
        }
    __syncthreads();
    const int n_rows_all = a.batch * a.num_q_heads * a.q_len;
    for (int e = tid; e < nr * Dv; e += kWT) {
        const int r = e / Dv, dv = e - r * Dv;
        float l = 0.f;
        for (int w2 = 0; w2 < kWWaves; ++w2) l += red2[w2 * RP + r];
        float o = 0.f;
        for (int s2 = 0; s2 < kWWaves; ++s2) o += obuf[((size_t)s2 * RP + r) * Dv + dv];
        float m = 0.f;
#pragma unroll
        for (int rr = 0; rr < RP; ++rr)
            if (rr == r) m = m_run[rr];
        const int row = r0 + r;
        const int g = row / a.q_len, qi = row - g * a.q_len;
        const int h = kv * p.G + g;
        const int rid = (b * a.num_q_heads + h) * a.q_len + qi;
        if (p.n_splits == 1) {
            ssq_store_elem(a.out, a.v_dtype, (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)qi * a.o_sl + dv, o / l);
            if (a.lse && dv == 0) a.lse[rid] = m + logf(l);
        } else {
            p.ws_o[((size_t)split * n_rows_all + rid) * Dv + dv] = o;
            if (dv == 0) {
                p.ws_m[(size_t)split * n_rows_all + rid] = m;
                p.ws_l[(size_t)split * n_rows_all + rid] = l;
            }
        }
    }
}

template <int RP, bool PAGED, int VT, int TPT>
int launch_wide_t(const SsqGenericParams& dp, int n_groups, hipStream_t st) {
    auto kern = k_decode_wide<RP, PAGED, VT, 4, TPT, 4>;
    if (dp.a.block_dim == 4) {
        if (dp.a.n_blocks <= 16) kern = k_decode_wide<RP, PAGED, VT, 4, TPT, 2>;
    } else {
        kern = dp.a.n_blocks <= 16 ? k_decode_wide<RP, PAGED, VT, 2, TPT, 2> : k_decode_wide<RP, PAGED, VT, 2, TPT, 4>;
    }
    int rc = ssq_allow_lds((const void*)kern, (int)kMaxSmem, "hipFuncSetAttribute(decode wide)");
    if (rc) return rc;
    const size_t smem = wide_lds(dp.a, RP, TPT).total * sizeof(float);
    if (smem > kMaxSmem) return ssq_fail(SSQ_ERR_UNSUPPORTED, "staged-codebook decode: %zu bytes of LDS", smem);
    dim3 grid(dp.n_splits, n_groups, dp.a.batch * dp.a.num_kv_heads);
    hipLaunchKernelGGL(kern, grid, dim3(kWT), smem, st, dp);
    return ssq_check_hip(hipGetLastError(), "k_decode_wide launch");
}

template <int RP, bool PAGED, int VT>
int launch_wide_tpt(const SsqGenericParams& dp, int n_groups, hipStream_t st) {
    switch (wide_tpt(dp.split_len)) {
        case 2: return launch_wide_t<RP, PAGED, VT, 2>(dp, n_groups, st);
        default: return launch_wide_t<RP, PAGED, VT, 4>(dp, n_groups, st);
    }
}

template <int RP>
int launch_wide_rp(const SsqGenericParams& dp, int n_groups, hipStream_t st) {
    const bool paged = dp.a.layout == SSQ_PAGED;
    if (dp.a.v_dtype == SSQ_BF16)
        return paged ? launch_wide_tpt<RP, true, SSQ_BF16>(dp, n_groups, st)
                     : launch_wide_tpt<RP, false, SSQ_BF16>(dp, n_groups, st);
    return paged ? launch_wide_tpt<RP, true, SSQ_F16>(dp, n_groups, st)
                 : launch_wide_tpt<RP, false, SSQ_F16>(dp, n_groups, st);
}

// rows per workgroup: 1, 2 or 4 (the matrix-core blocks hold 4 rows either way; the softmax does not)
int wide_rows(int RP) { return RP <= 2 ? RP : 4; }

}  // namespace

// LDS bytes of the largest super-tile
size_t ssq_decode_wide_smem(const ssq_decode_args& a, int RP) {
    return wide_lds(a, wide_rows(RP), 4).total * sizeof(float);
}

bool ssq_decode_wide_fits(const ssq_decode_args& a) {
    const size_t ncb = (size_t)a.n_centroids * a.block_dim;
    return (a.block_dim == 2 || a.block_dim == 4) && ncb % 4 == 0 && ncb / 4 <= (size_t)kStagePieces * kWT &&
           (a.value_dim == 64 || a.value_dim == 128) &&
           (a.v_dtype == SSQ_BF16 || a.v_dtype == SSQ_F16);
}

int ssq_decode_wide(const SsqGenericParams& dp, int RP, int n_groups, size_t, hipStream_t st) {
    switch (wide_rows(RP)) {
        case 1: return launch_wide_rp<1>(dp, n_groups, st);
        case 2: return launch_wide_rp<2>(dp, n_groups, st);
        default: return launch_wide_rp<4>(dp, n_groups, st);
    }
}
