// Nearest-codeword encode on the matrix cores (SunShapeBlockCodec.quantize, sunshape/codec.py:362-385):
// a bf16 MFMA screen finds, per (key, block), the one group of 8 or 16 codewords that can hold the
// reference's winner, and the reference's own fp32 arithmetic decides inside it.  Serves 256-codeword
// codebooks (kernel 2) and, with the codebook streamed through LDS, codebooks past 256 codewords.
//
// Screen.  v_mfma_f32_32x32x16_bf16 with codewords as rows and keys as columns evaluates
//   v_j = |c_j|^2 - 2 x.c_j + X_up = |x - c_j|^2 + (X_up - |x|^2),   X_up = |x|^2 rounded up to bf16.
// Every fp32 number enters as a sum of bf16 parts (RNE, each the rounding of what the previous left):
//   bf16 keys (and fp32 keys whose low halves are all zero):  x . (c_hi + c_mid + c_lo), exact products;
//   other keys:  x_hi (c_hi + c_mid) + x_mid c_hi, which leaves out at most 3 2^-18 |x||c| per product;
//   block dims 1 and 2, any key:  the six products down to 2^-18, which leave out less than 2^-25 |x||c|;
//   |c|^2 in three parts against 1, X_up against 1.
// That is 3 bd + 4 (6 bd + 4) of the K slots: one MFMA for block dims up to 4, two for 8, four for 16.
// v_j >= 0 up to rounding, so its bits order as a signed int.
//
// What it replaces and why.  The fp32 form (v_mfma_f32_16x16x4f32, K = bd + 2 padded to 8) spent 64
// matrix-core cycles per 256 distances and three VALU instructions per distance on the lane's two
// smallest values.  Here a 32x32 tile takes 32 cycles per 1,024 distances, and the VALU takes
// v_min3_i32 over each group of 8 codewords (16 past 256 codewords) before the tagged (min, second
// min) pair sees it: 7 instructions per 8 distances (11 per 16).  The exact evaluation then takes half
// a group on each of a key's two lanes.
//
// Measured, one MI355X, the fp32 screen / exact scan before -> this kernel: 262,144 bf16 keys of head_dim
// 128 at block_dim 4, 256 codewords: 625 -> 164 us (77 MB, 15 us at a copy's rate: VALU issue bounds it,
// 288 VALU instructions per 32 keys and block at 73 % issue, the matrix cores 13 % busy); 65,536 fp32
// keys at 4,096 codewords of dim 4: 1,448 -> 375 us; a 64-sequence decode step's append: unchanged,
// 11 us.
//
// Error bound.  P_j = (|x| + |c_j|)^2.  The terms of v_j pass through at most as many
// roundings (any order, even truncation) of partial sums of at most 1.02 P_j, |c_j|^2 carries the
// bd roundings of the reference's own norm, and the parts left out add 1.53 2^-18 P_j (2^-24):
// |v_j - (|x - c_j|^2 + X_up - |x|^2)| <= A P_j.  The reference's chain r_j is within g P_j of
// |x - c_j|^2, g = 1.001 (bd + 2) 2^-23.  With |c_j| <= |x| + |x - c_j|, P_j <= 6 |x|^2 + 3 |x - c_j|^2.
// The reference's winner j* has sqrt(r_j*) <= sqrt(r_m) for the screen's minimum m, and a correctly
// rounded sqrt merges values at most 2^-21 apart, so with S = max(v_m - (X_up - |x|^2), 0) and
// B = A + g,
//   v_j* <= v_m + 2^-20 S + 2 B (6 |x|^2 + 3 (1.01 S + 64 B |x|^2))
//        <= v_m + (2^-20 + 6.2 B) S + 12.6 B |x|^2         (B < 2^-15).
// thr adds 2^-17 relative for the tag bits (at most 2^-18 of v_m) and 2^-100 for underflow.  Every
// codeword that can win has v <= thr, so when one group alone reaches thr the winner is in it.
// Otherwise (and for keys or codewords whose squares pass 2^120 or are not finite, and when two
// candidates' distances are too close for their square roots to be told apart) the wave evaluates
// every codeword of the block for that key.  The code is therefore the reference's, whatever the
// matrix core's rounding order.
#include "ssq_encode_math.h"

#include <string.h>

#include <type_traits>

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef uint16_t __attribute__((may_alias)) u16a;
typedef uint32_t __attribute__((may_alias)) u32a;

// 16 waves x 32 keys: four waves per SIMD, so one wave's LDS and matrix-core latencies hide behind
// the others' minima, and the 256 codewords' operand is built once per 512 keys.
constexpr int kTileWaves = 16;
constexpr int kTileThreads = kTileWaves * SSQ_WAVE;
constexpr int kTileKeys = kTileWaves * 32;
// keys per slot of the staged keys, padded by one: consecutive slots then start two banks apart
constexpr int kKeyRow = kTileKeys + 1;
// Codewords per group: 8 where each block of 256 pays for the exact evaluation of a group; 16 past
// that, where the screen is nearly all of it (11 instructions per 16 distances instead of 14).
constexpr int group_cw(bool wide) { return wide ? 16 : 8; }
// tiles per (min, second min) pair: 16 group tags
constexpr int tag_tiles(bool wide) { return group_cw(wide); }
// codewords per LDS stage: a 256-codeword block, or 1,024 (block dim 8: 512) codewords of a longer one
constexpr int stage_cw(int bdp, bool wide) { return !wide ? 256 : bdp <= 4 ? 1024 : 512; }
constexpr size_t kTileSmemCap = 160 * 1024;
constexpr int kMaxLightTile = 128;

enum { kKeyBf16 = 0, kKeyF16 = 1, kKeyF32 = 2 };

struct TileParams {
    ssq_encode_args a;
    float ex[2], es[2];  // thr's |x|^2 and S factors: [0] keys exact in one bf16 part, [1] two-part keys
    int nbc;             // light blocks per workgroup chunk
    int n_light, chunks, fold;
    int xg, groups;      // key groups per (sequence, KV head), and in all
    int row_codes;       // 1: one chunk holds every light block and code rows take 16-byte stores
    int vec;             // 1: codeword rows are aligned for vector loads
    int pieces;          // 16-byte pieces per key row where rows load whole (a power of two), else 0
    uint8_t light[kMaxLightTile];  // light (VQ-coded) block ids, ascending
};

template <int BDP, bool WIDE>
struct TileShape {
    static constexpr int kNorm = BDP == 2 ? 6 : 3 * BDP / 2;         // operand dword of the norm's parts
    static constexpr int NM = (2 * (kNorm + 2) + 15) / 16;           // MFMAs per tile
    static constexpr int kTiles = stage_cw(BDP, WIDE) / 32;
    static constexpr int kOps = kTiles * NM * 256;                   // dwords of one stage's codeword operand
    static constexpr int kRec = 4 * BDP + 4;                         // 4 codewords and their norms (dwords)
    static constexpr int kRecs = WIDE ? 0 : stage_cw(BDP, WIDE) / 4 * kRec;
};
constexpr int slot_dwords(int bdp, bool raw16) { return raw16 ? bdp / 2 : bdp; }

// (key, block) pairs a workgroup can put off to its end (the full scans); more are scanned at once
constexpr int kOpenCap = 512;

// LDS: operands [2][kOps] | (one stage only: records [2][kRecs]) | bad [nbc], two-part flag, open
//      count | slot of block [128] | heavy blocks [128] | open pairs [kOpenCap] u16 | (under a
//      metric: E_b [nbc][BDP][BDP]) | keys [nbc + 1][kKeyRow][slot dwords] (the last slot takes
//      the dims of other chunks and of heavy blocks where rows load whole; block dims 9 and 10 are
//      always gathered and have none)
template <int BDP, bool WIDE>
size_t tile_smem(int nbc, bool raw16, const ssq_encode_args& a) {
    using Sh = TileShape<BDP, WIDE>;
    const size_t dw = 2 * (size_t)Sh::kOps + 2 * (size_t)Sh::kRecs + (size_t)((nbc + 5) & ~3) + 64 + kOpenCap / 2;
    return (dw + (a.metric ? (size_t)nbc * BDP * BDP : 0) + (size_t)(nbc + (BDP < 16 ? 1 : 0)) * kKeyRow * slot_dwords(BDP, raw16)) * 4 + 16;
}

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
    const v2f f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2bf));
}
// both values' bf16 roundings, packed, and what they leave
__device__ __forceinline__ uint32_t split2(float v0, float v1, float& r0, float& r1) {
    const uint32_t w = pk_bf16(v0, v1);
    r0 = v0 - __uint_as_float(w << 16);
    r1 = v1 - __uint_as_float(w & 0xFFFF0000u);
    return w;
}

// this lane's value and that of the lane 32 apart, in an order that differs between the two: only
// symmetric combinations are taken
__device__ __forceinline__ void pair32(int v, int& a, int& b) {
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    a = (int)r[0];
    b = (int)r[1];
}
// median of three signed ints (no builtin exposes v_med3_i32); operands are VALU results
__device__ __forceinline__ int med3_s(int a, int b, int c) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

template <int BDP>
__device__ __forceinline__ float norm_p(const float (&v)[BDP]) {  // sq_norm; zero padding is neutral
    float s = v[0] * v[0];
#pragma unroll
    for (int d = 1; d < BDP; ++d) {
        const float t = v[d] * v[d];
        s = s + t;
    }
    return s;
}
// the reference chain over [-2x, |x|^2, 1] . [c, 1, |c|^2], clamped at 0 (NaN: 0)
template <int BDP>
__device__ __forceinline__ float exact_e(const float (&m2x)[BDP], float xn, const float (&c)[BDP], float cn) {
    float acc = m2x[0] * c[0];
#pragma unroll
    for (int d = 1; d < BDP; ++d) acc = __builtin_fmaf(m2x[d], c[d], acc);
    acc = __builtin_fmaf(xn, 1.0f, acc);
    acc = __builtin_fmaf(1.0f, cn, acc);
    return fmaxf(acc, 0.f);
}

// the two smallest of a set of clamped distances (as their bits: values >= 0 order like ints), and
// the smallest one's index
constexpr int kInfBits = 0x7F800000;
struct Top2 {
    int e1, e2, n;
};
__device__ __forceinline__ Top2 join(const Top2& a, const Top2& b) {
    Top2 r;
    r.n = b.e1 < a.e1 ? b.n : a.n;
    r.e1 = min(a.e1, b.e1);
    r.e2 = min(min(a.e2, b.e2), max(a.e1, b.e1));
    return r;
}

// N consecutive dwords of LDS, as wide as their alignment (N dwords, at most 16 bytes) allows
template <int N>
__device__ __forceinline__ void lds_dwords(const u32a* s, uint32_t (&w)[N]) {
    if constexpr (N == 1) {
        w[0] = s[0];
    } else if constexpr (N == 2) {
        const uint2 v = *reinterpret_cast<const uint2*>(s);
        w[0] = v.x; w[1] = v.y;
    } else {
        static_assert(N % 4 == 0, "whole 16-byte pieces");
#pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            const uint4 v = reinterpret_cast<const uint4*>(s)[i];
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
        }
    }
}

// key elements of one slot as fp32
template <int BDP, int KM>
__device__ __forceinline__ void slot_elems(const uint32_t (&w)[slot_dwords(BDP, KM != kKeyF32)], float (&x)[BDP]) {
    if constexpr (KM == kKeyF32) {
#pragma unroll
        for (int d = 0; d < BDP; ++d) x[d] = __uint_as_float(w[d]);
    } else {
#pragma unroll
        for (int d = 0; d < BDP / 2; ++d) {
            x[2 * d] = KM == kKeyBf16 ? __uint_as_float(w[d] << 16) : ssq_f16_to_f32(w[d] & 0xFFFFu);
            x[2 * d + 1] = KM == kKeyBf16 ? __uint_as_float(w[d] & 0xFFFF0000u) : ssq_f16_to_f32(w[d] >> 16);
        }
    }
}

// the codeword row j of a block (zero-padded to BDP), in the metric space when met is given
template <int BDP>
__device__ __forceinline__ void load_row(const float* cent, uint32_t j, int bd, int vec, float (&c)[BDP]) {
    const float* s = cent + j * (uint32_t)bd;  // at most 2^20 rows of 16: a 32-bit offset from a uniform base
    if (vec) {  // bd == BDP
        if constexpr (BDP == 2) {
            const float2 v = *reinterpret_cast<const float2*>(s);
            c[0] = v.x; c[1] = v.y;
        } else {
#pragma unroll
            for (int q = 0; q < BDP / 4; ++q) {
                const float4 v = reinterpret_cast<const float4*>(s)[q];
                c[4 * q] = v.x; c[4 * q + 1] = v.y; c[4 * q + 2] = v.z; c[4 * q + 3] = v.w;
            }
        }
    } else {
#pragma unroll
        for (int d = 0; d < BDP; ++d) c[d] = s[min(d, bd - 1)];
#pragma unroll
        for (int d = 0; d < BDP; ++d) c[d] = d < bd ? c[d] : 0.f;
    }
}
// y_k = sum_j E_b[k][j] v_j (metric_row's order), in place; eb: E_b in LDS, zero-padded like v
template <int BDP>
__device__ __forceinline__ void to_metric(const float* eb, float (&v)[BDP]) {
    float y[BDP];
#pragma unroll
    for (int k = 0; k < BDP; ++k) {
        y[k] = eb[k * BDP] * v[0];
#pragma unroll
        for (int j = 1; j < BDP; ++j) y[k] = __builtin_fmaf(eb[k * BDP + j], v[j], y[k]);
    }
#pragma unroll
    for (int k = 0; k < BDP; ++k) v[k] = y[k];
}

__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// BDP: the block dim padded to 2, 4, 8 or 16 (zeros, neutral in every sum above).  KM: how the keys
// are staged: their 16 bits, or fp32 (also the metric images of 16-bit keys).  WIDE: more than one
// stage of codewords per block.
template <int BDP, int KM, bool WIDE>
__global__ __launch_bounds__(kTileThreads) void k_encode_tile(const TileParams p) {
    using Sh = TileShape<BDP, WIDE>;
    constexpr int NM = Sh::NM, kNorm = Sh::kNorm, kGc = group_cw(WIDE), kTagTiles = tag_tiles(WIDE);
    constexpr int SD = slot_dwords(BDP, KM != kKeyF32);
    extern __shared__ __align__(16) uint32_t tile_lds[];
    const ssq_encode_args& a = p.a;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;

    // workgroup -> (key group, block chunk): the chunks of one key group go to one XCD, one after
    // another, so the key rows they all read are in its L2
    const int id = blockIdx.x;
    const int chunk = (id >> 3) % p.chunks;
    const int g = ((id >> 3) / p.chunks) * 8 + (id & 7);
    if (g >= p.groups) return;
    const int y = g / p.xg;
    const SsqKeyMap km(a, p.fold, p.fold ? y : y % a.num_kv_heads, p.fold ? 0 : y / a.num_kv_heads);
    const int kv = km.kv, n_keys = km.n_keys;
    const int s0 = (g - y * p.xg) * kTileKeys + wave * 32;  // this wave's first key
    const bool live = s0 < n_keys;                          // wave-uniform
    const int l0 = chunk * p.nbc;
    const int nl = min(p.nbc, p.n_light - l0);
    const int bd = a.block_dim, D = a.head_dim, nb = a.n_blocks, nc = a.n_centroids;
    const uint64_t hm0 = a.heavy_mask[0], hm1 = a.heavy_mask[1];
    const bool do_heavy = chunk == 0 && (hm0 | hm1);

    u32a* ops = tile_lds;
    u32a* recs = ops + 2 * Sh::kOps;
    u32a* bad = recs + 2 * Sh::kRecs;
    u32a* two_part = bad + p.nbc;
    uint32_t* n_open = tile_lds + 2 * Sh::kOps + 2 * Sh::kRecs + p.nbc + 1;
    uint8_t* blkslot = reinterpret_cast<uint8_t*>(bad + ((p.nbc + 5) & ~3));
    uint8_t* heavyL = blkslot + 128;
    u16a* open_list = reinterpret_cast<u16a*>(heavyL + 128);
    float* metL = reinterpret_cast<float*>(open_list + kOpenCap);  // [nl][BDP][BDP]
    u32a* keysL = reinterpret_cast<u32a*>(open_list + kOpenCap) + (a.metric ? p.nbc * BDP * BDP : 0);
    u32a* mykeys = keysL + (wave * 32) * SD;  // slot j of key m: mykeys + (j * kKeyRow + m) * SD

    for (int j = tid; j <= p.nbc + 1; j += kTileThreads) bad[j] = 0;  // and *two_part, *n_open
    if (tid < nb) {
        const bool hv = ssq_is_heavy(hm0, hm1, tid);
        const int ho = heavy_ordinal(hm0, hm1, tid);
        if (hv) heavyL[ho] = (uint8_t)tid;
        const int li = tid - ho - l0;  // ordinal among this chunk's light blocks
        blkslot[tid] = hv || li < 0 || li >= nl ? 255 : (uint8_t)li;
    }

    const float* cent = a.cent + (int64_t)kv * a.cent_sh;
    const int64_t* perm = a.perm + (int64_t)kv * a.perm_sh;
    const float* met = a.metric ? a.metric + (int64_t)kv * a.metric_sh : nullptr;

    if (met) {  // the chunk's diagonal blocks of the metric
        for (int i = tid; i < nl * BDP * BDP; i += kTileThreads) {
            const int r = i / BDP % BDP, c = i % BDP;
            const int64_t o = p.light[l0 + i / (BDP * BDP)] * bd;
            metL[i] = r < bd && c < bd ? met[(o + r) * D + o + c] : 0.f;
        }
    }

    // output rows of this lane's key, and the row of its elements
    int64_t crow = 0, prow = 0, krow = 0;
    if (live) {
        int b, s;
        km.bs(a, min(s0 + col, n_keys - 1), b, s);
        krow = (int64_t)b * a.k_sb + (int64_t)kv * a.k_sh + (int64_t)s * a.k_ss;
        out_rows(a, b, kv, s, crow, prow);
    }

    // keys -> LDS, permuted: slot j holds light block l0 + j's elements.
    //  Whole rows: each lane loads 16-byte pieces of several keys, always the same dims, and scatters
    //  the elements to the byte offsets the inverse permutation gives for those dims (an LDS table,
    //  in the operand buffers' space): no arithmetic per element.
    //  Otherwise (unaligned rows, padded block dims, a permutation that repeats a dim): a lane takes
    //  one element position, its dim from the permutation, of 64 / epad keys at a time.
    uint32_t low = 0;  // any nonzero low half of an fp32 element
    const int E = nl * BDP;
    int pieces = p.pieces;
    if (pieces) {  // uniform
        constexpr int kElem = KM == kKeyF32 ? 4 : 2;
        constexpr int N = 8;  // pieces in flight per lane; the first ones load while the table is built
        uint4 v[N];
        const int pc = lane & (pieces - 1), m0 = lane / pieces, kpl = 64 / pieces, n_loads = pieces / 2;
        auto load_pieces = [&](int i0) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int m = min(i0 + i, n_loads - 1) * kpl + m0;
                const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)krow, m);
                const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)((uint64_t)krow >> 32), m);
                const int64_t row = (int64_t)(((uint64_t)hi << 32) | lo);
                v[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(a.keys) + row * kElem + pc * 16);
            }
        };
        if (live) load_pieces(0);
        const uint32_t other = (uint32_t)(p.nbc * kKeyRow * SD * 4);
        for (int d = tid; d < D; d += kTileThreads) ops[d] = other;
        __syncthreads();  // also: bad and *two_part are cleared
        auto dim_of = [&](int e) { return (int)perm[p.light[l0 + e / BDP] * bd + e % BDP]; };
        auto off_of = [&](int e) { return (uint32_t)((e / BDP) * kKeyRow * SD * 4 + (e % BDP) * kElem); };
        for (int e = tid; e < E; e += kTileThreads) {
            const int dim = dim_of(e);
            if ((unsigned)dim < (unsigned)D) ops[dim] = off_of(e);
        }
        __syncthreads();
        for (int e = tid; e < E; e += kTileThreads) {
            const int dim = dim_of(e);
            if ((unsigned)dim >= (unsigned)D || ops[dim] != off_of(e)) *two_part = 2;  // a dim twice
        }
        __syncthreads();
        const bool twice = *two_part == 2;
        constexpr int kPer = 16 / kElem;  // elements per piece
        uint32_t off[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) off[k] = ops[pc * kPer + k];
        __syncthreads();  // the table's space becomes the operand buffers, the flag the two-part flag
        if (twice) pieces = 0;
        if (tid == 0) *two_part = 0;
        if (pieces && live) {
            for (int i0 = 0; i0 < n_loads; i0 += N) {
                if (i0) load_pieces(i0);
                char* dst = reinterpret_cast<char*>(mykeys + m0 * SD) + i0 * kpl * SD * 4;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    if (i0 + i >= n_loads) break;  // uniform
                    const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if constexpr (KM == kKeyF32) {
                            *reinterpret_cast<u32a*>(dst + off[k]) = w[k];
                            low |= w[k] & 0xFFFFu;
                        } else {
                            *reinterpret_cast<u16a*>(dst + off[2 * k]) = (uint16_t)w[k];
                            *reinterpret_cast<u16a*>(dst + off[2 * k + 1]) = (uint16_t)(w[k] >> 16);
                        }
                    }
                    dst += kpl * SD * 4;
                }
            }
            wave_sync_lds();
        }
    }
    if constexpr (KM == kKeyF32) __syncthreads();  // *two_part is cleared
    if (live && !pieces) {
        int epad = BDP;
        while (epad < E && epad < 64) epad <<= 1;
        const int sub = lane / epad, kp = 64 / epad, trips = 32 / kp;
        for (int e0 = 0; e0 < E; e0 += epad) {
            const int e = e0 + (lane & (epad - 1));
            const int j = e / BDP, d = e - j * BDP;
            const bool in = j < nl;
            const bool real = in && d < bd;
            const int64_t dim = real ? perm[p.light[l0 + j] * bd + d] : 0;
            auto take = [&](int m0, auto count) {  // count keys per lane, their loads in flight together
                constexpr int N = decltype(count)::value;
                int64_t at[N];
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const int m = (m0 + i) * kp + sub;
                    const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)krow, m);
                    const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)((uint64_t)krow >> 32), m);
                    at[i] = (int64_t)(((uint64_t)hi << 32) | lo) + dim;
                }
                if constexpr (KM == kKeyF32) {
                    float v[N];
                    ssq_load_elems<N>(a.keys, a.k_dtype, at, v);
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        const int m = (m0 + i) * kp + sub;
                        const uint32_t u = real ? __float_as_uint(v[i]) : 0u;
                        low |= u & 0xFFFFu;
                        if (in) mykeys[(j * kKeyRow + m) * SD + d] = u;
                    }
                } else {
                    uint32_t v[N];
#pragma unroll
                    for (int i = 0; i < N; ++i) v[i] = reinterpret_cast<const uint16_t*>(a.keys)[at[i]];
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        const int m = (m0 + i) * kp + sub;
                        if (in)
                            reinterpret_cast<u16a*>(mykeys + (j * kKeyRow + m) * SD)[d] = real ? (uint16_t)v[i] : (uint16_t)0;
                    }
                }
            };
            if (trips >= 8)
                for (int m0 = 0; m0 < trips; m0 += 8) take(m0, std::integral_constant<int, 8>{});
            else
                for (int m0 = 0; m0 < trips; ++m0) take(m0, std::integral_constant<int, 1>{});
        }
        wave_sync_lds();
    }
    if (met) __syncthreads();  // metL
    if (KM == kKeyF32 && met && live) {  // the key blocks' images under the block metric
        low = 0;
        for (int j = half; j < nl; j += 2) {
            u32a* ks = mykeys + (j * kKeyRow + col) * SD;
            uint32_t kw[SD];
            float x[BDP];
            lds_dwords<SD>(ks, kw);
            slot_elems<BDP, KM>(kw, x);
            to_metric<BDP>(metL + j * BDP * BDP, x);
#pragma unroll
            for (int d = 0; d < BDP; ++d) {
                ks[d] = __float_as_uint(x[d]);
                low |= __float_as_uint(x[d]) & 0xFFFFu;
            }
        }
        wave_sync_lds();
    }
    // whether every key of the workgroup is exact in one bf16 part
    if (KM == kKeyF32 && low) *two_part = 1;
    __syncthreads();
    const bool one_part = BDP == 2 || KM == kKeyBf16 || (KM == kKeyF32 && *two_part == 0);
    const float ex = one_part ? p.ex[0] : p.ex[1], es = one_part ? p.es[0] : p.es[1];

    // A stage's codewords, one per thread: with 1,024-codeword stages every wave builds, with smaller
    // ones the waves take turns.  The rows load two stages ahead; the operand is written at the start
    // of the stage before it, beside the other waves' work.  (A quarter codeword per thread, so that
    // every wave builds 256-codeword stages too, took more instructions in all: 188 against 169 us.)
    constexpr int kSc = stage_cw(BDP, WIDE), kTurns = kTileThreads / kSc;
    const int nst = WIDE ? (nc + kSc - 1) / kSc : 1;
    const int n_it = nl * nst;
    const int bcw = tid & (kSc - 1);
    float cw[BDP];
    auto builds = [&](int it) { return it < n_it && wave / (kTileWaves / kTurns) == (it & (kTurns - 1)); };
    int lj = 0, lst = 0;  // block and stage of the next load
    auto load_next = [&](int it) {
        if (builds(it)) {
            const float* cb = cent + (int64_t)p.light[l0 + lj] * nc * bd;
            load_row<BDP>(cb, min(lst * kSc + bcw, nc - 1), bd, p.vec, cw);
        }
        if (++lst == nst) { lst = 0; ++lj; }
    };
    // operand dword i of a codeword, from its row's first dword: [MFMA][half][row][4 dwords]
    constexpr auto at_dw = [](int i) { return (i / 8) * 256 + ((i / 4) & 1) * 128 + (i & 3); };
    auto store_cw = [&](int it, int j, int st) {
        if (met) to_metric<BDP>(metL + j * BDP * BDP, cw);
        const float cn = norm_p<BDP>(cw);
        if (!(cn < 0x1.0p120f)) bad[j] = 1;
        uint32_t kd[8 * NM];
#pragma unroll
        for (int i = 0; i < 8 * NM; ++i) kd[i] = 0;
#pragma unroll
        for (int d = 0; d < BDP; d += 2) {
            float r0, r1, s0, s1;
            const uint32_t hw = split2(-2.0f * cw[d], -2.0f * cw[d + 1], r0, r1);
            const uint32_t mw = split2(r0, r1, s0, s1), lw = pk_bf16(s0, s1);
            if constexpr (BDP == 2) {
                kd[0] = kd[2] = kd[5] = hw;
                kd[1] = kd[4] = mw;
                kd[3] = lw;
            } else {
                kd[d / 2] = hw;
                kd[(BDP + d) / 2] = mw;
                kd[(2 * BDP + d) / 2] = one_part ? lw : hw;
            }
        }
        float r1, u, r2;
        split2(cn, 0.f, r1, u);
        kd[kNorm] = split2(cn, r1, u, r2);
        kd[kNorm + 1] = pk_bf16(r2, 1.0f);
        if (WIDE && st * kSc + bcw >= nc) {  // past the codebook's end: 2^126, larger than any threshold
#pragma unroll
            for (int i = 0; i < 8 * NM; ++i) kd[i] = i == kNorm ? 0x7E80u : 0u;
        }
        // row of codeword w of its tile: a lane's 16 accumulators are then 16 consecutive codewords
        const int w = bcw & 31;
        const int row = 8 * ((w >> 2) & 3) + 4 * (w >> 4) + (w & 3);
        u32a* dst = ops + (it & 1) * Sh::kOps + (bcw >> 5) * NM * 256 + row * 4;
#pragma unroll
        for (int i = 0; i < 8 * NM; i += 4)
            *reinterpret_cast<uint4*>(dst + at_dw(i)) = make_uint4(kd[i], kd[i + 1], kd[i + 2], kd[i + 3]);
        if constexpr (!WIDE) {
            u32a* rec = recs + (it & 1) * Sh::kRecs + (bcw >> 2) * Sh::kRec;
#pragma unroll
            for (int d = 0; d < BDP; ++d) rec[(bcw & 3) * BDP + d] = __float_as_uint(cw[d]);
            rec[4 * BDP + (bcw & 3)] = __float_as_uint(cn);
        }
    };
    // every codeword of block j for key kk of the workgroup, over the lanes of a wave: the reference's
    // chain, the first index of the smallest sqrt.  A wave busy with it holds the whole workgroup at
    // the next barrier (it takes longer than a 256-codeword block), so the open pairs wait for the
    // end, where the lanes share them, and this serves only those past the list's end.
    auto scan_all = [&](int j, int kk) {
        u32a* ks = keysL + (j * kKeyRow + kk) * SD;
        uint32_t kwm[SD];
        float xm[BDP];
        lds_dwords<SD>(ks, kwm);
        slot_elems<BDP, KM>(kwm, xm);
        const float xmn = norm_p<BDP>(xm);
#pragma unroll
        for (int d = 0; d < BDP; ++d) xm[d] = -2.0f * xm[d];
        const int blk = p.light[l0 + j];
        const float* cb = cent + (int64_t)blk * nc * bd;
        float be = INFINITY;  // the smallest clamped value, and the first index of its sqrt
        uint32_t bn = 0x7FFFFFFFu;
        constexpr int NB = BDP <= 4 ? 4 : BDP <= 8 ? 2 : 1;
#pragma unroll 1
        for (int n0 = lane; n0 < nc; n0 += 64 * NB) {
            float c[NB][BDP];
#pragma unroll
            for (int i = 0; i < NB; ++i) load_row<BDP>(cb, min(n0 + 64 * i, nc - 1), bd, p.vec, c[i]);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                if (met) to_metric<BDP>(metL + j * BDP * BDP, c[i]);
                // past the end: the last codeword again, which cannot win over itself
                take_min(exact_e<BDP>(xm, xmn, c[i], norm_p<BDP>(c[i])), (uint32_t)min(n0 + 64 * i, nc - 1), be, bn);
            }
        }
        if (bn == 0x7FFFFFFFu) bn = (uint32_t)lane;  // every value infinite
        float bf = __builtin_sqrtf(be);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float of = __shfl_xor(bf, o);
            const uint32_t on = (uint32_t)__shfl_xor((int)bn, o);
            if (of < bf || (of == bf && on < bn)) { bf = of; bn = on; }
        }
        if (lane == 0) ks[0] = bn;
        wave_sync_lds();
    };

    load_next(0);
    if (builds(0)) store_cw(0, 0, 0);
    load_next(1);
    __syncthreads();

    for (int j = 0, it = 0; j < nl; ++j) {
        u32a* ks = mykeys + (j * kKeyRow + col) * SD;
        uint32_t kw[SD];
        float x[BDP];
        float xn = 0.f, dlt = 0.f;
        v8bf kb[NM];
        if (live) {
            // the key's operand: [hi, hi, hi or mid, 1, 1, 1, X_up]
            lds_dwords<SD>(ks, kw);
            slot_elems<BDP, KM>(kw, x);
            xn = norm_p<BDP>(x);
            const uint32_t xu = (__float_as_uint(xn) + 0xFFFFu) & 0xFFFF0000u;
            dlt = __uint_as_float(xu) - xn;
            uint32_t kd[8 * NM];
#pragma unroll
            for (int i = 0; i < 8 * NM; ++i) kd[i] = 0;
            if constexpr (BDP == 2) {
                if constexpr (KM == kKeyBf16) {
                    kd[0] = kd[1] = kd[3] = kw[0];
                } else {
                    float r0, r1, t0, t1;
                    kd[0] = kd[1] = kd[3] = split2(x[0], x[1], r0, r1);
                    kd[2] = kd[4] = split2(r0, r1, t0, t1);
                    kd[5] = pk_bf16(t0, t1);
                }
            } else
#pragma unroll
            for (int d = 0; d < BDP; d += 2) {
                uint32_t hw, third;
                if constexpr (KM == kKeyBf16) {
                    hw = third = kw[d / 2];
                } else {
                    float r0, r1;
                    hw = split2(x[d], x[d + 1], r0, r1);
                    third = one_part ? hw : pk_bf16(r0, r1);
                }
                kd[d / 2] = hw;
                kd[(BDP + d) / 2] = hw;
                kd[(2 * BDP + d) / 2] = third;
            }
            kd[kNorm] = 0x3F803F80u;
            kd[kNorm + 1] = 0x3F80u | xu;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                uint4 v;
                v.x = half ? kd[8 * m + 4] : kd[8 * m];
                v.y = half ? kd[8 * m + 5] : kd[8 * m + 1];
                v.z = half ? kd[8 * m + 6] : kd[8 * m + 2];
                v.w = half ? kd[8 * m + 7] : kd[8 * m + 3];
                kb[m] = __builtin_bit_cast(v8bf, v);
            }
        }
        int m1 = 0x7FFFFFFF, m2 = 0x7FFFFFFF, mst = 0;
        for (int st = 0; st < nst; ++st, ++it) {
            if (builds(it + 1)) store_cw(it + 1, st + 1 == nst ? j + 1 : j, st + 1 == nst ? 0 : st + 1);
            load_next(it + 2);
            if (live) {
                // Tile t + 1's MFMA is issued before tile t's minima are taken, and its operand read
                // a tile earlier still (the scheduling barriers keep that order).
                const u32a* op = ops + (it & 1) * Sh::kOps + lane * 4;
                auto opnd = [&](int t, int m) {
                    return __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4*>(op + (t * NM + m) * 256));
                };
                v8bf av[2][NM];
                v16f acc[2];
                auto issue = [&](int t) {
                    v16f c = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int m = 0; m < NM; ++m) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[t & 1][m], kb[m], c, 0, 0, 0);
                    acc[t & 1] = c;
                };
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    av[0][m] = opnd(0, m);
                    av[1][m] = opnd(1, m);
                }
                issue(0);
                int q1 = 0x7FFFFFFF, q2 = 0x7FFFFFFF;
#pragma unroll
                for (int t = 0; t < Sh::kTiles; ++t) {
                    if (t + 2 < Sh::kTiles) {
#pragma unroll
                        for (int m = 0; m < NM; ++m) av[t & 1][m] = opnd(t + 2, m);
                    }
                    if (t + 1 < Sh::kTiles) issue(t + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int u = 0; u < 16 / kGc; ++u) {  // codewords 32 t + 16 half + kGc u ... + kGc - 1
                        int b[kGc];
#pragma unroll
                        for (int i = 0; i < kGc; ++i) b[i] = __float_as_int(acc[t & 1][kGc * u + i]);
                        int v = min(min(b[0], b[1]), b[2]);  // v_min3_i32
#pragma unroll
                        for (int i = 3; i + 1 < kGc; i += 2) v = min(min(v, b[i]), b[i + 1]);
                        v = min(v, b[kGc - 1]);
                        v = (v & -16) | ((16 / kGc) * (t % kTagTiles) + u);
                        q2 = med3_s(q1, q2, v);
                        q1 = min(q1, v);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (WIDE) {
                        if (t % kTagTiles == kTagTiles - 1) {
                            m2 = min(min(max(m1, q1), m2), q2);
                            mst = q1 < m1 ? st * (Sh::kTiles / kTagTiles) + t / kTagTiles : mst;
                            m1 = min(m1, q1);
                            q1 = q2 = 0x7FFFFFFF;
                        }
                    }
                }
                if constexpr (!WIDE) {
                    m1 = q1;
                    m2 = q2;
                }
            }
            if (live && (!WIDE || st + 1 == nst)) {
                // threshold from the key's minimum (its tag in the low bits), and whether one group
                // alone reaches it.  Bit l of the masks below is key l; a key's other lane is 32 bits up.
                int pa, pb;
                pair32((m1 & -32) | ((m1 & 15) << 1) | half, pa, pb);
                const int pk = min(pa, pb);
                const float mt = fmaxf(__int_as_float(pk & -32), 0.f) * (1.0f + 0x1.0p-17f);
                const float thr = mt + es * fmaxf(mt - dlt, 0.f) + ex * xn + 0x1.0p-100f;
                const uint64_t b1 = __builtin_amdgcn_ballot_w64(__int_as_float(m1 & -32) <= thr);
                const uint64_t b2 = __builtin_amdgcn_ballot_w64(__int_as_float(m2 & -32) <= thr);
                const uint64_t fin = __builtin_amdgcn_ballot_w64(xn < 0x1.0p120f);
                uint32_t ok = (uint32_t)fin & (uint32_t)(b1 ^ (b1 >> 32)) & ~(uint32_t)(b2 | (b2 >> 32));
                if (__builtin_amdgcn_readfirstlane(bad[j])) ok = 0;
                float m2x[BDP];
#pragma unroll
                for (int d = 0; d < BDP; ++d) m2x[d] = -2.0f * x[d];
                // the reference's arithmetic inside the group: half of its codewords on each of the key's lanes
                constexpr int NC = kGc / 2;
                const int tag = (pk >> 1) & 15;
                int first = (WIDE ? tag * 32 : (tag >> 1) * 32 + (tag & 1) * 8) + (pk & 1) * 16 + half * NC;
                Top2 best[NC];
                if constexpr (WIDE) {
                    int sa, sb;
                    pair32(m1, pa, pb);
                    pair32(mst, sa, sb);
                    first += (pa < pb ? sa : sb) * (32 * kTagTiles);
                    const int blk = p.light[l0 + j];
                    const float* cb = cent + (int64_t)blk * nc * bd;
                    float c[NC][BDP];
#pragma unroll
                    for (int i = 0; i < NC; ++i) load_row<BDP>(cb, min(first + i, nc - 1), bd, p.vec, c[i]);
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        if (met) to_metric<BDP>(metL + j * BDP * BDP, c[i]);
                        const float e = exact_e<BDP>(m2x, xn, c[i], norm_p<BDP>(c[i]));
                        best[i] = {first + i < nc ? __float_as_int(e) : kInfBits, kInfBits, i};
                    }
                } else {
                    uint32_t rec[Sh::kRec];
                    lds_dwords<Sh::kRec>(recs + (it & 1) * Sh::kRecs + (first >> 2) * Sh::kRec, rec);
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        float c[BDP];
#pragma unroll
                        for (int d = 0; d < BDP; ++d) c[d] = __uint_as_float(rec[i * BDP + d]);
                        const float e = exact_e<BDP>(m2x, xn, c, __uint_as_float(rec[4 * BDP + i]));
                        best[i] = {__float_as_int(e), kInfBits, i};
                    }
                }
#pragma unroll
                for (int w = 1; w < NC; w <<= 1)
#pragma unroll
                    for (int i = 0; i < NC; i += 2 * w) best[i] = join(best[i], best[i + w]);
                int ea, eb;
                pair32(best[0].e1, ea, eb);
                const int e1 = min(ea, eb);
                const bool mine = best[0].e1 == e1;
                const float e2 = __int_as_float(mine ? best[0].e2 : best[0].e1);
                const uint64_t bm = __builtin_amdgcn_ballot_w64(mine);
                // below t the smaller value's correctly rounded sqrt is the smaller one
                const uint64_t far = __builtin_amdgcn_ballot_w64(__int_as_float(e1) < e2 * 0x1.ffffep-1f - 0x1.0p-146f);
                ok &= (uint32_t)(far & (far >> 32)) & (uint32_t)(bm ^ (bm >> 32));
                // the code takes the place of the block's key elements
                if (mine && ((ok >> col) & 1)) ks[0] = (uint32_t)(first + best[0].n);
                const uint32_t todo = ~ok;
                if (todo) {  // rare: to the list for the end; what does not fit there is scanned here
                    int at = 0;
                    if (lane == 0) at = (int)atomicAdd(n_open, (uint32_t)__popc(todo));
                    at = __builtin_amdgcn_readfirstlane(at);
                    const int pos = at + __popc(todo & ((1u << col) - 1u));
                    if (half == 0 && ((todo >> col) & 1) && pos < kOpenCap)
                        open_list[pos] = (uint16_t)(j * kTileKeys + wave * 32 + col);
                    if (at + __popc(todo) > kOpenCap) {
                        wave_sync_lds();
                        for (uint32_t t = todo; t; t &= t - 1)
                            if (at++ >= kOpenCap) scan_all(j, wave * 32 + __builtin_ctz(t));
                    }
                }
                wave_sync_lds();
            }
            __syncthreads();
        }
    }
    // The pairs put off, published by the loop's last barrier: 16 lanes per 256 codewords of a pair,
    // 16 codewords a lane; (sqrt bits, index) pairs meet in a 64-bit LDS minimum, which orders them as
    // the reference does (the operand buffers' space).
    const int n_put = nl > 0 ? min((int)__builtin_amdgcn_readfirstlane(*n_open), kOpenCap) : 0;
    if (n_put) {
        unsigned long long* res = reinterpret_cast<unsigned long long*>(tile_lds);
        if (tid < n_put) res[tid] = ~0ull;
        __syncthreads();
        const int parts = (nc + 255) / 256;
        for (int i = tid >> 4; i < n_put * parts; i += kTileThreads / 16) {
            const int en = i / parts, n1 = (i - en * parts) * 256 + (tid & 15);
            const int j = open_list[en] / kTileKeys;
            uint32_t kwm[SD];
            float xm[BDP];
            lds_dwords<SD>(keysL + (j * kKeyRow + open_list[en] % kTileKeys) * SD, kwm);
            slot_elems<BDP, KM>(kwm, xm);
            const float xmn = norm_p<BDP>(xm);
#pragma unroll
            for (int d = 0; d < BDP; ++d) xm[d] = -2.0f * xm[d];
            const int blk = p.light[l0 + j];
            const float* cb = cent + (int64_t)blk * nc * bd;
            float be = INFINITY;
            uint32_t bn = 0x7FFFFFFFu;
            constexpr int NB = BDP <= 4 ? 16 : BDP <= 8 ? 4 : 1;
#pragma unroll 1
            for (int n0 = n1; n0 < n1 + 256; n0 += 16 * NB) {
                float c[NB][BDP];
#pragma unroll
                for (int u = 0; u < NB; ++u) load_row<BDP>(cb, min(n0 + 16 * u, nc - 1), bd, p.vec, c[u]);
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    if (met) to_metric<BDP>(metL + j * BDP * BDP, c[u]);
                    take_min(exact_e<BDP>(xm, xmn, c[u], norm_p<BDP>(c[u])), (uint32_t)min(n0 + 16 * u, nc - 1), be, bn);
                }
            }
            if (bn == 0x7FFFFFFFu) bn = (uint32_t)min(n1, nc - 1);  // every value infinite
            atomicMin(&res[en], ((unsigned long long)__float_as_uint(__builtin_sqrtf(be)) << 32) | bn);
        }
        __syncthreads();
        if (tid < n_put) {
            const int j = open_list[tid] / kTileKeys;
            keysL[(j * kKeyRow + open_list[tid] % kTileKeys) * SD] = (uint32_t)res[tid];
        }
        __syncthreads();
    }
    if (!live) return;

    // codes out: whole rows in 16-byte pieces, or element by element; lane and lane + 32 share a key
    const bool mine = s0 + col < n_keys;
    const int cwid = ssq_code_width(nc);
    const u32a* ck = mykeys + col * SD;
    if (p.row_codes) {
        const int per = 16 / cwid, pieces = nb / per;
        if (mine) {
            for (int q = half; q < pieces; q += 2) {
                uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    if (i >= per) break;
                    const int sl = blkslot[q * per + i];
                    const uint32_t c = sl == 255 ? 0u : ck[sl * kKeyRow * SD];
                    if (cwid == 1) w[i >> 2] |= c << (8 * (i & 3));
                    else if (cwid == 2) w[(i >> 1) & 3] |= c << (16 * (i & 1));
                    else w[i & 3] = c;
                }
                *reinterpret_cast<uint4*>(a.codes + (crow * cwid + 16 * q)) = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
    } else if (mine) {
        for (int j = half; j < nl; j += 2) store_code(a.codes, cwid, crow + p.light[l0 + j], ck[j * kKeyRow * SD]);
        if (do_heavy) {
            const int nh = __popcll(hm0) + __popcll(hm1);
            for (int i = half; i < nh; i += 2) store_code(a.codes, cwid, crow + heavyL[i], 0u);
        }
    }
    if (do_heavy && mine) {  // passthrough values (sunshape/codec.py:367-372)
        const int nh = __popcll(hm0) + __popcll(hm1);
        const int n = nh * bd;
        constexpr int N = 8;
        for (int e0 = half; e0 < n; e0 += 2 * N) {
            int64_t at[N];
            float v[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int e = min(e0 + 2 * i, n - 1);
                const int o = e / bd;
                at[i] = krow + perm[heavyL[o] * bd + (e - o * bd)];
            }
            ssq_load_elems<N>(a.keys, a.k_dtype, at, v);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int e = e0 + 2 * i;
                if (e < n) {
                    const int o = e / bd;
                    const int slot = a.pt_dense ? heavyL[o] : o;
                    ssq_store_elem(a.pt, a.pt_dtype, prow + (int64_t)slot * bd + (e - o * bd), v[i]);
                }
            }
        }
    }
}

template <int BDP, int KM, bool WIDE>
int launch_tile(TileParams& tp, hipStream_t st) {
    const ssq_encode_args& a = tp.a;
    constexpr bool raw16 = KM != kKeyF32;
    int nbc = tp.n_light > 0 ? tp.n_light : 1;
    while (nbc > 1 && tile_smem<BDP, WIDE>(nbc, raw16, a) > kTileSmemCap) --nbc;
    tp.fold = ssq_encode_fold(&a, kTileKeys);
    const int64_t n_keys = tp.fold ? (int64_t)a.batch * a.seq_len : a.seq_len;
    const int64_t xg = (n_keys + kTileKeys - 1) / kTileKeys;
    const int64_t groups = xg * (tp.fold ? a.num_kv_heads : (int64_t)a.batch * a.num_kv_heads);
    // Smaller chunks of blocks until the workgroups fill the chip: a few keys (a decode step's
    // append) take one block per workgroup.  Past 256 codewords a block is long, so the chunks
    // shrink until there are two workgroups per CU to even out the last round.
    const int64_t want_wg = (WIDE ? 2 : 1) * (int64_t)ssq_device_cus();
    if (tp.n_light > 0) {
        int chunks = (tp.n_light + nbc - 1) / nbc;
        if (groups * chunks < want_wg) {
            const int64_t want = (want_wg + groups - 1) / groups;
            chunks = (int)(want < tp.n_light ? want : tp.n_light);
        }
        nbc = (tp.n_light + chunks - 1) / chunks;
    }
    tp.nbc = nbc;
    tp.chunks = tp.n_light > 0 ? (tp.n_light + nbc - 1) / nbc : 1;
    // whole key rows in 16-byte pieces: chunks that use most of a row, aligned rows in the staged
    // type, pieces that divide a wave
    const int elem = raw16 ? 2 : 4;
    const int pieces = a.head_dim * elem / 16;
    const bool staged_type = raw16 || a.k_dtype == SSQ_F32;
    tp.pieces = BDP < 16 && 2 * nbc * BDP > a.head_dim && a.block_dim == BDP && staged_type && (a.head_dim * elem) % 16 == 0 && pieces >= 2 && pieces <= 64 &&
                        (pieces & (pieces - 1)) == 0 && (uintptr_t)a.keys % 16 == 0 && (a.k_sb * elem) % 16 == 0 &&
                        (a.k_sh * elem) % 16 == 0 && (a.k_ss * elem) % 16 == 0
                    ? pieces
                    : 0;
    const int cw = ssq_code_width(a.n_centroids);
    tp.row_codes = tp.chunks == 1 && (a.n_blocks * cw) % 16 == 0 && (uintptr_t)a.codes % 16 == 0 &&
                   (a.c_sb * cw) % 16 == 0 && (a.c_sh * cw) % 16 == 0 && (a.c_st * cw) % 16 == 0;
    const int64_t wgs = 8 * ((groups + 7) / 8) * tp.chunks;
    SSQ_UNSUPPORTED(groups <= 0x7fffffff && wgs <= 0x7fffffff, "too many keys for one encode launch");
    tp.xg = (int)xg;
    tp.groups = (int)groups;
    const size_t smem = tile_smem<BDP, WIDE>(nbc, raw16, a);
    SSQ_UNSUPPORTED(smem <= kTileSmemCap, "block too large for the MFMA encode");
    const int rc = ssq_allow_lds((const void*)k_encode_tile<BDP, KM, WIDE>, (int)kTileSmemCap,
                                 "hipFuncSetAttribute(encode tile)");
    if (rc) return rc;
    hipLaunchKernelGGL((k_encode_tile<BDP, KM, WIDE>), dim3((unsigned)wgs), dim3(kTileThreads), smem, st, tp);
    return ssq_check_hip(hipGetLastError(), "k_encode_tile launch");
}

template <int BDP, bool WIDE>
int launch_tile_keys(TileParams& tp, hipStream_t st) {
    const ssq_encode_args& a = tp.a;
    if (a.k_dtype == SSQ_F32 || a.metric) return launch_tile<BDP, kKeyF32, WIDE>(tp, st);
    if (a.k_dtype == SSQ_BF16) return launch_tile<BDP, kKeyBf16, WIDE>(tp, st);
    return launch_tile<BDP, kKeyF16, WIDE>(tp, st);
}

}  // namespace

int ssq_encode_tile_run(const ssq_encode_args* a, hipStream_t st) {
    TileParams tp;
    memset(&tp, 0, sizeof(tp));
    tp.a = *a;
    const int bd = a->block_dim;
    for (int two = 0; two < 2; ++two) {  // the bound of the file comment, rounded up
        const double gr = 1.001 * (bd + 2) * 0x1.0p-23;
        const int terms = (bd <= 2 ? 6 : 3) * bd + 4;
        const double left = bd <= 2 ? 0x1.0p-24 : two ? 1.53 * 0x1.0p-18 : 0.0;
        const double A = 1.02 * terms * 0x1.0p-23 + bd * 0x1.0p-24 + left;
        const double B = A + gr;
        tp.ex[two] = (float)(12.6 * B * 1.001);
        tp.es[two] = (float)((0x1.0p-20 + 6.2 * B) * 1.001);
    }
    for (int blk = 0; blk < a->n_blocks; ++blk) {
        const bool heavy = blk < 64 ? ((a->heavy_mask[0] >> blk) & 1) : ((a->heavy_mask[1] >> (blk - 64)) & 1);
        if (!heavy) tp.light[tp.n_light++] = (uint8_t)blk;
    }
    const int64_t al = bd == 2 ? 8 : 16;
    tp.vec = (bd == 2 || bd == 4 || bd == 8 || bd == 16) && (uintptr_t)a->cent % al == 0 && (a->cent_sh * 4) % al == 0;
    const bool wide = a->n_centroids > 256;
    const int bdp = bd <= 2 ? 2 : bd <= 4 ? 4 : bd <= 8 ? 8 : 16;
    switch (bdp * 2 + (wide ? 1 : 0)) {
        case 4: return launch_tile_keys<2, false>(tp, st);
        case 5: return launch_tile_keys<2, true>(tp, st);
        case 8: return launch_tile_keys<4, false>(tp, st);
        case 9: return launch_tile_keys<4, true>(tp, st);
        case 16: return launch_tile_keys<8, false>(tp, st);
        case 17: return launch_tile_keys<8, true>(tp, st);
        default: return launch_tile_keys<16, false>(tp, st);  // block dims 9 and 10, 256 codewords
    }
}
