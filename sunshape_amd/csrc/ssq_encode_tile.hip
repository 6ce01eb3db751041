// Nearest-codeword encode on the matrix cores (SunShapeBlockCodec.quantize, sunshape/codec.py:362-385):
// a bf16 MFMA screen finds, per (key, block), the one group of 8 or 16 codewords that can hold the
// reference's winner, and the reference's own fp32 arithmetic decides inside it.  Serves 256-codeword
// codebooks (kernel 2) and, with the codebook streamed through LDS, codebooks past 256 codewords.
//
// Screen.  With mu a point near the middle of the block's codebook, c' = c - mu and n = |c'|^2 + 2 mu.c',
// v_mfma_f32_32x32x16_bf16 with codewords as rows and keys as columns evaluates
//   v_j = n_j - 2 x.c'_j + X_up = |x - c_j|^2 + (X_up - |x - mu|^2),   X_up = |x - mu|^2 rounded up to bf16.
// Every fp32 number enters as a sum of bf16 parts (RNE, each the rounding of what the previous left):
//   bf16 keys (and fp32 keys whose low halves are all zero):  x . (c'_hi + c'_mid + c'_lo), exact products;
//   block dims 1 and 2, any key:  the six products down to 2^-18, which leave out less than 2^-25 |x||c'|;
//   other keys, with x' = x - mu in place of x and n = |c'|^2:  x'_hi (c'_hi + c'_mid) + x'_mid c'_hi, which
//   leaves out at most 3 2^-18 |x'||c'| per product;
//   n in three parts against 1, X_up against 1.
// That is 3 bd + 4 (6 bd + 4) of the K slots: one MFMA for block dims up to 4, two for 8, four for 16.
// v_j >= 0 up to rounding, so its bits order as a signed int.  (bf16 keys keep their own bits, as x - mu
// is no bf16 number.)  No product is larger than |x||c'|, so an offset that keys and codewords share, as K
// projections have per channel, weighs on the error bound once and not squared.
//
// What it replaces and why.  The fp32 form (v_mfma_f32_16x16x4f32, K = bd + 2 padded to 8) spent 64
// matrix-core cycles per 256 distances and three VALU instructions per distance on the lane's two
// smallest values.  Here a 32x32 tile takes 32 cycles per 1,024 distances, and the VALU takes
// v_min3_i32 over each group of 8 codewords (16 past 256 codewords) before the tagged (min, second
// min) pair sees it: 7 instructions per 8 distances (11 per 16).  The exact evaluation then takes half
// a group on each of a key's two lanes.
//
// Measured, one MI355X, the fp32 screen / exact scan before -> this kernel: 262,144 bf16 keys of head_dim
// 128 at block_dim 4, 256 codewords: 631 -> 184 us (77 MB, 15 us at a copy's rate: VALU issue bounds it,
// 283 VALU instructions per 32 keys and block in 68 % of the issue slots, the matrix cores 15 % busy);
// 65,536 fp32 keys at 4,096 codewords of dim 4, with the dequantize's 26: 1,434 -> 404 us (VALU 82 %,
// matrix cores 32 %); a 64-sequence decode step's append: 13.4 -> 13.1 us with the call.
// Keys and codewords that share an offset of 0, 10, 30 and 100 standard deviations, bf16, 8 heads: 8,192 rows
// at 256 codewords of dim 4: 59, 61, 76 and 205 us (the fp32 screen 168, 204, 257 and 439; with |x|^2 in this
// screen's bound 54, 94, 546 and 977); 4,096 rows at 4,096 codewords: 205, 304, 718 and 1,035 (the exact scan
// 735).  Slower than what they replaced: codebooks past 256 codewords around the last offset, or that hold
// every codeword twice (1.1 to 1.4 times, at 300 codewords 1.8), and block_dim 1 for at most 128 keys (10 to
// 35 %, 1 to 5 us).
//
// Error bound.  d_j = |x - c_j|, y = |x - mu|, m = |mu|; |c'_j| <= y + d_j.  The terms of v_j pass through
// at most as many roundings (any order, even truncation) of partial sums of at most
// 1.02 (|c'|^2 + 2 (m + |x|) |c'| + 1.01 y^2); n carries 2 bd roundings of its own, c' and x' one each, and
// the parts left out add L |x||c'|, L = 6.16 2^-18 (0 for keys exact in one part).  So with
// A = 1.02 terms 2^-23 + (2 bd + 2) 2^-24,
//   |v_j - (d_j^2 + X_up - y^2)| <= A (2.51 y^2 + 3 d_j^2 + 2 (m + |x|) (y + d_j)) + L |x| (y + d_j),
// and for two-part keys the same with y for |x| and 0 for m.
// The reference's chain r_j = ((-2x.c_j) + |x|^2) + |c_j|^2 rounds its product's bd steps at most at
// 2 |x||c_j|, the first sum at d_j^2 + |c_j|^2 and the second at d_j^2, and |c_j|^2 carries bd roundings;
// the roundings of |x|^2 are the same for every j.  Beside those it is within G_j of d_j^2, with
// g = 1.01 2^-24 and |c_j| <= |x| + d_j,
//   G_j <= g (2 bd |x||c_j| + (bd + 1) |c_j|^2 + 2 d_j^2) <= g ((3.13 bd + 1.07) |x|^2 + (33 bd + 19) d_j^2).
// The reference's winner j* has sqrt(r_j*) <= sqrt(r_m) (negative r: 0, which adds no more than the
// roundings of |x|^2, at most bd g |x|^2) for the screen's minimum m, and a correctly rounded sqrt merges
// values at most 2^-21 apart, so with S = max(v_m - (X_up - y^2), 0), both d_j*^2 and d_m^2 are at most
// Q = 1.03 S + 20 (A + L + 2 g (3.13 bd + 1.07)) (|x|^2 + y^2), and
//   v_j* <= v_m + 5.02 A y^2 + 2 g (3.13 bd + 1.07) |x|^2 + (6 A + 2 g (33 bd + 19) + 2^-20) Q
//               + (4 A m + (4 A + 2 L) |x|) sqrt(2 (y^2 + Q)),   m <= |x| + y;
// where mu is 0 (y = |x|), the last term is at most (4 A + 2 L) (1.4143 |x|^2 + 0.7072 Q).
// thr adds 2^-17 relative for the tag bits (at most 2^-18 of v_m) and 2^-100 for underflow.  Every
// codeword that can win has v <= thr, so when one group alone reaches thr the winner is in it.
// Otherwise (and for keys or codewords whose squares pass 2^120 or are not finite, and when two
// candidates' distances are too close for their square roots to be told apart) every codeword of the
// block is evaluated for that key: such pairs go to a list that the whole workgroup scans at its end, 16
// lanes a pair, or, where a block leaves many, to a scan of the block from LDS.  The code is
// therefore the reference's, whatever the matrix core's rounding order.
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

// factors of the file comment's threshold
struct ScreenBound {
    float s, a, x;    // S, |x - mu|^2, |x|^2
    float qa, qs, qx;  // |x - mu|^2, S, |x|^2 inside the square root that bounds |x - mu| + |x - c|
    float m, n;       // |mu|, |x| (two-part keys: |x - mu|) times that root
    float cs, cx;     // S, |x|^2 where mu is 0
};

struct TileParams {
    ssq_encode_args a;
    ScreenBound bound[2];  // [0] keys exact in one bf16 part, [1] two-part keys
    int nbc;             // light blocks per workgroup chunk
    int n_light, chunks, fold;
    int xg, groups;      // key groups per (sequence, KV head), and in all
    int row_codes;       // 1: one chunk holds every light block and code rows take 16-byte stores
    int vec;             // 1: codeword rows are aligned for vector loads
    int center;          // 0: mu is 0
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

// (key, block) pairs that a workgroup can put off: to its end, or (256 codewords) until kOpenFlush are
// waiting after a block.  A block that leaves more than open_block of its 512 keys open is scanned for
// all of them at once (scan_block): one pair costs 1.6 times as much on the list, where a lane reads each
// codeword from memory, at 256 codewords, 3.5 at 4,096 and 7 at 16,384.  Once two blocks and at
// least half of those so far failed (of a chunk of at most 8 blocks: the first one, with more than
// kOpenMost open), the screen ends and the rest are scanned.
constexpr int kOpenCap = 1024;
constexpr int kOpenFlush = 512;
__device__ __forceinline__ int open_block(int nc) { return nc <= 256 ? 256 : nc <= 8192 ? 128 : 64; }
constexpr int kOpenMost = kTileKeys / 2;

// mu costs a small call up to 1 us and saves it little: few open pairs have the whole workgroup (block
// dims 9 and 10, whose scans are the longest, take it at every size)
constexpr int kCenterKeys = 64;

// LDS: operands [2][kOps] | (one stage only: records [2][kRecs]) | bad [nbc] (1: not finite, 4: mu is not 0, 2: failed), two-part flag, open
//      count, failed [2], a block's open count [3], unused | mu [nbc][BDP] | decided keys
//      [nbc][kTileWaves] | slot of block [128] | heavy blocks [128] | open pairs [kOpenCap] u16 | (under a
//      metric: E_b [nbc][BDP][BDP]) | keys [nbc (+ 1)][kKeyRow][slot dwords]: where rows load whole, the
//      last slot takes the dims of other chunks and of heavy blocks (a chunk of every dim has none of
//      them, and block dims 9 and 10 are always gathered)
template <int BDP, bool WIDE>
size_t tile_smem(int nbc, bool raw16, const ssq_encode_args& a) {
    using Sh = TileShape<BDP, WIDE>;
    const size_t dw = 2 * (size_t)Sh::kOps + 2 * (size_t)Sh::kRecs + (size_t)((nbc + 11) & ~3) +
                      (size_t)((nbc * BDP + 3) & ~3) + (size_t)nbc * kTileWaves + 64 + kOpenCap / 2;
    const int slots = nbc + (BDP < 16 && nbc * BDP != a.head_dim ? 1 : 0);
    return (dw + (a.metric ? (size_t)nbc * BDP * BDP : 0) + (size_t)slots * kKeyRow * slot_dwords(BDP, raw16)) * 4 + 16;
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
    uint32_t* badA = tile_lds + 2 * Sh::kOps + 2 * Sh::kRecs;
    uint32_t* n_open = tile_lds + 2 * Sh::kOps + 2 * Sh::kRecs + p.nbc + 1;
    uint32_t* failed = n_open + 1;  // [parity of the block]
    uint32_t* n_blk = failed + 2;   // [block modulo 3]
    u32a* muL = bad + ((p.nbc + 11) & ~3);
    u32a* okL = muL + ((p.nbc * BDP + 3) & ~3);
    uint8_t* blkslot = reinterpret_cast<uint8_t*>(okL + p.nbc * kTileWaves);
    uint8_t* heavyL = blkslot + 128;
    u16a* open_list = reinterpret_cast<u16a*>(heavyL + 128);
    float* metL = reinterpret_cast<float*>(open_list + kOpenCap);  // [nl][BDP][BDP]
    u32a* keysL = reinterpret_cast<u32a*>(open_list + kOpenCap) + (a.metric ? p.nbc * BDP * BDP : 0);
    u32a* mykeys = keysL + (wave * 32) * SD;  // slot j of key m: mykeys + (j * kKeyRow + m) * SD

    for (int j = tid; j < p.nbc + 7; j += kTileThreads) bad[j] = 0;  // and *two_part, *n_open, failed, n_blk
    for (int j = tid; j < p.nbc * kTileWaves; j += kTileThreads) okL[j] = ~0u;
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

    // Loads whose use comes after the keys': the chunk's diagonal blocks of the metric, and for mu, the mean
    // of 16 codewords spread over a block's codebook, one dim of them per lane.
    if (met) {
        for (int i = tid; i < nl * BDP * BDP; i += kTileThreads) {
            const int r = i / BDP % BDP, c = i % BDP;
            const int64_t o = p.light[l0 + i / (BDP * BDP)] * bd;
            metL[i] = r < bd && c < bd ? met[(o + r) * D + o + c] : 0.f;
        }
    }
    float mc[16];
    auto load_mean = [&](int i) {
        const float* cb = cent + (int64_t)p.light[l0 + i / BDP] * nc * bd + min(i % BDP, bd - 1);
#pragma unroll
        for (int u = 0; u < 16; ++u) mc[u] = cb[((uint32_t)(u * nc) >> 4) * (uint32_t)bd];
    };
    if (p.center && tid < nl * BDP) load_mean(tid);

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
    if (p.center || met) __syncthreads();  // metL, and bad is cleared
    // mu: 0 where the codebook is centred already (or not finite)
    for (int i = tid; p.center && i < nl * BDP; i += kTileThreads) {
        if (i >= kTileThreads) load_mean(i);
        const int d = i % BDP;
        float m = 0.f, q = 0.f;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            m += mc[u];
            q = __builtin_fmaf(mc[u], mc[u], q);
        }
        m = d < bd ? m * 0.0625f : 0.f;
        q = d < bd ? q * 0.0625f : 0.f;
        float m2 = m * m;
#pragma unroll
        for (int o = 1; o < BDP; o <<= 1) {
            m2 += __shfl_xor(m2, o);
            q += __shfl_xor(q, o);
        }
        m = m2 > 0.25f * q ? m : 0.f;
        if (met) {  // its image
            float y = 0.f;
#pragma unroll
            for (int c = 0; c < BDP; ++c) y = __builtin_fmaf(metL[i * BDP + c], __shfl(m, (lane & ~(BDP - 1)) + c), y);
            m = y;
        }
        muL[i] = __float_as_uint(m);
        if (m != 0.f) bad[i / BDP] = 4;
    }
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
    const ScreenBound& bound = p.bound[one_part ? 0 : 1];

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
        if (!(cn < 0x1.0p120f)) atomicOr(&badA[j], 1u);
        float c[BDP], n = cn;  // the codeword from mu, and |c|^2 (+ 2 mu.c)
#pragma unroll
        for (int d = 0; d < BDP; ++d) c[d] = cw[d];
        if (__builtin_amdgcn_readfirstlane(bad[j]) & 4) {  // mu is not 0
            n = 0.f;
#pragma unroll
            for (int d = 0; d < BDP; ++d) {
                const float mu = __uint_as_float(muL[j * BDP + d]);
                c[d] = cw[d] - mu;
                n = __builtin_fmaf(__builtin_fmaf(one_part ? 2.0f : 0.0f, mu, c[d]), c[d], n);
            }
        }
        uint32_t kd[8 * NM];
#pragma unroll
        for (int i = 0; i < 8 * NM; ++i) kd[i] = 0;
#pragma unroll
        for (int d = 0; d < BDP; d += 2) {
            float r0, r1, s0, s1;
            const uint32_t hw = split2(-2.0f * c[d], -2.0f * c[d + 1], r0, r1);
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
        split2(n, 0.f, r1, u);
        kd[kNorm] = split2(n, r1, u, r2);
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
    // Codewords n1 + 16 i below n2 of a listed pair on one lane: (sqrt bits, index) of its first minimum,
    // which order as the reference does.
    auto scan_pair = [&](int pair, int n1, int n2, auto batch) {
        constexpr int NB = decltype(batch)::value;  // codewords in flight
        const int j = pair / kTileKeys;
        uint32_t kwm[SD];
        float xm[BDP];
        lds_dwords<SD>(keysL + (j * kKeyRow + pair % kTileKeys) * SD, kwm);
        slot_elems<BDP, KM>(kwm, xm);
        const float xmn = norm_p<BDP>(xm);
#pragma unroll
        for (int d = 0; d < BDP; ++d) xm[d] = -2.0f * xm[d];
        const float* cb = cent + (int64_t)p.light[l0 + j] * nc * bd;
        float be = INFINITY;
        uint32_t bn = 0x7FFFFFFFu;
        bool in_lds = false;
        if constexpr (!WIDE) {  // a chunk of at most two blocks (a few keys) still has their records
            in_lds = nl <= 2;
            const u32a* rj = recs + (j & 1) * Sh::kRecs;
            for (int n = n1; in_lds && n < n2; n += 16) {
                const u32a* rec = rj + (n >> 2) * Sh::kRec;
                float c[BDP];
#pragma unroll
                for (int d = 0; d < BDP; ++d) c[d] = __uint_as_float(rec[(n & 3) * BDP + d]);
                take_min(exact_e<BDP>(xm, xmn, c, __uint_as_float(rec[4 * BDP + (n & 3)])), (uint32_t)n, be, bn);
            }
        }
#pragma unroll 1
        for (int n0 = in_lds ? n2 : n1; n0 < n2; n0 += 16 * NB) {
            float c[NB][BDP];
#pragma unroll
            for (int u = 0; u < NB; ++u) load_row<BDP>(cb, min(n0 + 16 * u, nc - 1), bd, p.vec, c[u]);
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                if (met) to_metric<BDP>(metL + j * BDP * BDP, c[u]);
                // past the end: the last codeword again, which cannot win over itself
                take_min(exact_e<BDP>(xm, xmn, c[u], norm_p<BDP>(c[u])), (uint32_t)min(n0 + 16 * u, nc - 1), be, bn);
            }
        }
        if (bn == 0x7FFFFFFFu) bn = (uint32_t)min(n1, nc - 1);  // every value infinite
        return ((unsigned long long)__float_as_uint(__builtin_sqrtf(be)) << 32) | bn;
    };
    auto put_code = [&](int pair, uint32_t n) { keysL[(pair / kTileKeys * kKeyRow + pair % kTileKeys) * SD] = n; };
    // the list, between two blocks (the whole workgroup): 16 lanes a pair
    auto scan_list = [&]() {
        const int n = min((int)__builtin_amdgcn_readfirstlane(*n_open), kOpenCap);
        for (int i = tid >> 4; i < n; i += kTileThreads / 16) {
            const int pair = open_list[i];
            if (bad[pair / kTileKeys] == 2) continue;
            unsigned long long r =
                scan_pair(pair, tid & 15, nc, std::integral_constant<int, BDP <= 4 ? 4 : BDP <= 8 ? 2 : 1>{});
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) {
                const unsigned long long t = ((unsigned long long)(uint32_t)__shfl_xor((int)(r >> 32), o) << 32) |
                                             (uint32_t)__shfl_xor((int)(uint32_t)r, o);
                r = t < r ? t : r;
            }
            if ((tid & 15) == 0) put_code(pair, (uint32_t)r);
        }
        __syncthreads();
        if (tid == 0) *n_open = 0;
    };
    // Every codeword of block j for its undecided keys (the whole workgroup; the operand buffers' space):
    // a stage's codewords and norms in LDS, half of them on each of a key's two lanes.
    auto scan_block = [&](int j) {
        constexpr int kBuf = kSc / 4 * Sh::kRec;
        static_assert(kBuf <= Sh::kOps, "a stage's records fit its operand");
        const int blk = p.light[l0 + j];
        const float* cb = cent + (int64_t)blk * nc * bd;
        const uint32_t need = live ? ~(uint32_t)__builtin_amdgcn_readfirstlane(okL[j * kTileWaves + wave]) : 0u;
        u32a* ks = mykeys + (j * kKeyRow + col) * SD;
        float m2x[BDP];
        {
            uint32_t kw[SD];
            lds_dwords<SD>(ks, kw);
            slot_elems<BDP, KM>(kw, m2x);
        }
        const float xn = norm_p<BDP>(m2x);
#pragma unroll
        for (int d = 0; d < BDP; ++d) m2x[d] = -2.0f * m2x[d];
        float be = INFINITY;
        uint32_t bn = (uint32_t)half;  // (every value infinite: the first index)
        float c[BDP];
        if (tid < kSc) load_row<BDP>(cb, min(tid, nc - 1), bd, p.vec, c);
        for (int st = 0; st < nst; ++st) {
            u32a* buf = ops + (st & 1) * kBuf;
            if (tid < kSc) {
                if (met) to_metric<BDP>(metL + j * BDP * BDP, c);
                u32a* rec = buf + (tid >> 2) * Sh::kRec;
#pragma unroll
                for (int d = 0; d < BDP; ++d) rec[(tid & 3) * BDP + d] = __float_as_uint(c[d]);
                rec[4 * BDP + (tid & 3)] = __float_as_uint(norm_p<BDP>(c));
                if (st + 1 < nst) load_row<BDP>(cb, min((st + 1) * kSc + tid, nc - 1), bd, p.vec, c);
            }
            __syncthreads();
            if (need) {
                // (past the end: the last codeword again, which cannot win over itself)
                constexpr int NR = BDP <= 4 ? 2 : 1;  // records whose distances are computed before their tests
                const int n_rec = (min(kSc, nc - st * kSc) + 3) / 4, mid = (n_rec / 2 + NR - 1) / NR * NR;
                const int g1 = half ? n_rec : mid;
                for (int g = half ? mid : 0; g < g1; g += NR) {
                    float e[4 * NR];
#pragma unroll
                    for (int r = 0; r < NR; ++r) {
                        uint32_t rec[Sh::kRec];
                        lds_dwords<Sh::kRec>(buf + (g + r) * Sh::kRec, rec);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float v = m2x[0] * __uint_as_float(rec[i * BDP]);
#pragma unroll
                            for (int d = 1; d < BDP; ++d) v = __builtin_fmaf(m2x[d], __uint_as_float(rec[i * BDP + d]), v);
                            v = __builtin_fmaf(xn, 1.0f, v);
                            e[4 * r + i] = __builtin_fmaf(1.0f, __uint_as_float(rec[4 * BDP + i]), v);
                        }
                    }
                    const int j0 = st * kSc + 4 * g;
#pragma unroll
                    for (int i = 0; i < 4 * NR; ++i) take_min(e[i], (uint32_t)min(j0 + i, nc - 1), be, bn);
                }
            }
        }
        __syncthreads();  // the buffers' last reads
        if (need) {
            const float bf = __builtin_sqrtf(be), of = __shfl_xor(bf, 32);
            const uint32_t on = (uint32_t)__shfl_xor((int)bn, 32);
            if (of < bf || (of == bf && on < bn)) bn = on;
            if (half == 0 && ((need >> col) & 1)) ks[0] = bn;
            wave_sync_lds();
        }
    };

    load_next(0);
    if (builds(0)) store_cw(0, 0, 0);
    load_next(1);
    __syncthreads();

    int n_fail = 0;
    for (int j = 0, it = 0, j3 = 0;; ++j, j3 = j3 == 2 ? 0 : j3 + 1) {
        u32a* ks = mykeys + (max(min(j, nl - 1), 0) * kKeyRow + col) * SD;
        uint32_t kw[SD];
        lds_dwords<SD>(ks, kw);
        const uint32_t bj = bad[j], fj = failed[(j & 1) ^ 1];  // (bad[nl] is a word of its own)
        // What the block before left open.  A wave of this block sets the other flag, and that one again
        // only after this block's barrier; the count of the next block is cleared meanwhile.
        const uint32_t fl = __builtin_amdgcn_readfirstlane(fj);
        if (fl) {  // uniform
            __syncthreads();
            if (tid == 0) failed[(j & 1) ^ 1] = 0;
            if (fl & 3) {
                ++n_fail;
                const bool quit = 2 * n_fail >= j && (n_fail >= 2 || ((fl & 2) && nl <= 8));
                for (int i = j - 1 + tid; i < (quit ? nl : j); i += kTileThreads) bad[i] = 2;
                if (quit) {
                    for (int i = j * kTileWaves + tid; i < nl * kTileWaves; i += kTileThreads) okL[i] = 0;
                    break;
                }
            }
            if constexpr (!WIDE) {
                if (fl & 4) {
                    __syncthreads();  // bad[j - 1]
                    scan_list();
                    __syncthreads();  // *n_open
                }
            }
        }
        if (j >= nl) break;
        if (tid == 0) n_blk[j3 == 2 ? 0 : j3 + 1] = 0;
        float x[BDP];
        float xn = 0.f, an = 0.f, dlt = 0.f;
        const bool off = __builtin_amdgcn_readfirstlane(bj) & 4;  // mu is not 0
        v8bf kb[NM];
        if (live) {
            // the key's operand: [hi, hi, hi or mid, 1, 1, 1, X_up]
            slot_elems<BDP, KM>(kw, x);
            xn = norm_p<BDP>(x);
            float xc[BDP];
#pragma unroll
            for (int d = 0; d < BDP; ++d) xc[d] = x[d];
            an = xn;
            if (off) {
#pragma unroll
                for (int d = 0; d < BDP; ++d) xc[d] = x[d] - __uint_as_float(muL[j * BDP + d]);
                an = norm_p<BDP>(xc);
            }
            const uint32_t xu = (__float_as_uint(an) + 0xFFFFu) & 0xFFFF0000u;
            dlt = __uint_as_float(xu) - an;
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
                    hw = split2(one_part ? x[d] : xc[d], one_part ? x[d + 1] : xc[d + 1], r0, r1);
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
                const float sm = fmaxf(mt - dlt, 0.f);
                float thr = mt + (bound.cs * sm + bound.cx * xn) + 0x1.0p-100f;
                if (off) {
                    const float root = __builtin_amdgcn_sqrtf(bound.qa * an + (bound.qs * sm + bound.qx * xn));
                    const float xr = __builtin_amdgcn_sqrtf(one_part ? xn : an), y = __builtin_amdgcn_sqrtf(an);
                    thr = mt + (bound.s * sm + bound.a * an + bound.x * xn) +
                          root * (bound.n * xr + bound.m * (xr + y)) + 0x1.0p-100f;  // m <= |x| + y
                }
                const uint64_t b1 = __builtin_amdgcn_ballot_w64(__int_as_float(m1 & -32) <= thr);
                const uint64_t b2 = __builtin_amdgcn_ballot_w64(__int_as_float(m2 & -32) <= thr);
                const uint64_t fin = __builtin_amdgcn_ballot_w64(xn < 0x1.0p120f);
                uint32_t ok = (uint32_t)fin & (uint32_t)(b1 ^ (b1 >> 32)) & ~(uint32_t)(b2 | (b2 >> 32));
                if (__builtin_amdgcn_readfirstlane(bad[j]) & 1) ok = 0;
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
                if (todo) {  // to the list, unless the block fails (scan_block then serves it)
                    const int n = __popc(todo);
                    int at = 0;
                    if (lane == 0) {
                        okL[j * kTileWaves + wave] = ok;
                        const int c = (int)atomicAdd(&n_blk[j3], (uint32_t)n) + n;
                        at = c > open_block(nc) ? kOpenCap : (int)atomicAdd(n_open, (uint32_t)n);
                        if (at + n > kOpenCap) atomicOr(&failed[j & 1], c > kOpenMost ? 3u : 1u);
                        else if (!WIDE && at + n > kOpenFlush) atomicOr(&failed[j & 1], 4u);
                    }
                    at = __builtin_amdgcn_readfirstlane(at);
                    const int pos = at + __popc(todo & ((1u << col) - 1u));
                    if (half == 0 && ((todo >> col) & 1) && pos < kOpenCap)
                        open_list[pos] = (uint16_t)(j * kTileKeys + wave * 32 + col);
                }
                wave_sync_lds();
            }
            __syncthreads();
        }
    }
    if (n_fail) {
        __syncthreads();
        for (int j = 0; j < nl; ++j)
            if (__builtin_amdgcn_readfirstlane(bad[j]) == 2) scan_block(j);
    }
    // The pairs on the list (published by the loop's last barrier; those of failed blocks are done): 16
    // lanes per 256 (block dims 9 and 10: 64) codewords of a pair; the results meet in a 64-bit LDS
    // minimum (the operand buffers' space).
    const int n_put = nl > 0 ? min((int)__builtin_amdgcn_readfirstlane(*n_open), kOpenCap) : 0;
    if (n_put) {
        unsigned long long* res = reinterpret_cast<unsigned long long*>(tile_lds);
        if (tid < n_put) res[tid] = ~0ull;
        __syncthreads();
        const int part = BDP == 16 ? 64 : 256, parts = (nc + part - 1) / part;
        for (int i = tid >> 4; i < n_put * parts; i += kTileThreads / 16) {
            const int en = i / parts, n1 = (i - en * parts) * part;
            const int pair = open_list[en];
            if (bad[pair / kTileKeys] == 2) continue;
            atomicMin(&res[en], scan_pair(pair, n1 + (tid & 15), n1 + part,
                                          std::integral_constant<int, BDP <= 4 ? 16 : BDP <= 8 ? 4 : 1>{}));
        }
        __syncthreads();
        if (tid < n_put && bad[open_list[tid] / kTileKeys] != 2) put_code(open_list[tid], (uint32_t)res[tid]);
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
    tp.center = n_keys > kCenterKeys || BDP == 16;
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
        const int terms = (bd <= 2 ? 6 : 3) * bd + 4;
        const double al = 1.02 * terms * 0x1.0p-23 + (2 * bd + 2) * 0x1.0p-24;
        const double left = bd <= 2 ? 0x1.0p-23 : two ? 6.16 * 0x1.0p-18 : 0.0;
        const double g = 1.01 * 0x1.0p-24, gx = 2 * g * (3.13 * bd + 1.07), gd = 2 * g * (33 * bd + 19);
        const double near = 6 * al + gd + 0x1.0p-20, k = 20 * (al + left + gx), up = 1.002;
        ScreenBound& b = tp.bound[two];
        b.s = (float)(1.03 * near * up);
        b.a = (float)((5.02 * al + near * k) * up);
        b.x = (float)((gx + near * k) * up);
        b.qa = (float)(2 * (1 + k) * up);
        b.qs = (float)(2.06 * up);
        b.qx = (float)(2 * k * up);
        b.m = (float)(bd > 2 && two ? 0.0 : 4 * al * up);
        b.n = (float)((4 * al + 2 * left) * up);
        const double cn = 4 * al + 2 * left;  // |x| sqrt(2 (|x|^2 + Q)) <= 1.4143 |x|^2 + 0.7072 Q
        b.cs = (float)(1.03 * (near + 0.7072 * cn) * up);
        b.cx = (float)((5.02 * al + gx + 1.4143 * cn + 2 * k * (near + 0.7072 * cn)) * up);
    }
    for (int blk = 0; blk < a->n_blocks; ++blk) {
        const bool heavy = blk < 64 ? ((a->heavy_mask[0] >> blk) & 1) : ((a->heavy_mask[1] >> (blk - 64)) & 1);
        if (!heavy) tp.light[tp.n_light++] = (uint8_t)blk;
    }
    const int64_t al = bd == 2 ? 8 : 16;
    tp.vec = (bd == 2 || bd == 4 || bd == 8 || bd == 16) && (uintptr_t)a->cent % al == 0 && (a->cent_sh * 4) % al == 0;
    const bool wide = a->n_centroids > 256;
    SSQ_UNSUPPORTED(!wide || (bd >= 3 && bd <= 8), "MFMA encode past 256 codewords needs block_dim 3 to 8");
    const int bdp = bd <= 2 ? 2 : bd <= 4 ? 4 : bd <= 8 ? 8 : 16;
    switch (bdp * 2 + (wide ? 1 : 0)) {
        case 4: return launch_tile_keys<2, false>(tp, st);
        case 8: return launch_tile_keys<4, false>(tp, st);
        case 9: return launch_tile_keys<4, true>(tp, st);
        case 16: return launch_tile_keys<8, false>(tp, st);
        case 17: return launch_tile_keys<8, true>(tp, st);
        default: return launch_tile_keys<16, false>(tp, st);  // block dims 9 and 10, 256 codewords
    }
}
