// Nearest-codeword encode (SunShapeBlockCodec.quantize, sunshape/codec.py:362-385).
//
// The reference picks, per block, argmin_c torch.cdist(x_b, C_b) with the first index on
// ties.  torch.cdist takes ATen's mm formulation for these sizes:
//   d2[c] = [-2x, |x|^2, 1] . [c, 1, |c|^2]   (fp32 GEMM, K = bd + 2, k ascending, FMA chain)
//   d[c]  = sqrt(max(d2[c], 0))
// with |v|^2 = left-to-right sum of rounded squares.  Every index this file returns is the
// first argmin of d computed with exactly that arithmetic and a correctly rounded sqrt.
// When both of cdist's inputs have at most 25 rows (a call that quantizes at most 25 keys with at
// most 25 codewords, e.g. 16 at 2 bits/dim and block_dim 2) torch evaluates the distance directly
// instead, d2[c] = sum_k (x_k - c_k)^2 with rounded squares summed in k order; the caller asks for
// that with direct_dist, which the exact scan serves.
//
// The entry point is here with k_encode_scan, one thread per (key, block) and the exact formula for
// every codeword.  256-codeword codebooks go to the matrix-core screen (ssq_encode_tile.hip), block
// dim 2 with a search grid to ssq_encode_grid.hip; codebooks past 256 codewords to the screen, or to
// the exact scan in ssq_encode_wide.hip.  Every kernel returns the same codes.
#include "ssq_encode_math.h"

#include <math.h>

namespace {

struct EncodeParams {
    ssq_encode_args a;
    int nbc;           // blocks per workgroup chunk
    int fold;          // short sequences: all sequences of a KV head share one key range (SsqKeyMap)
    int passes;        // key passes per workgroup (scan)
};

// ---------------------------------------------------------------------------
// exact scan: thread per (key, block); codebook chunk + norms in LDS
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 256;
constexpr int kScanPasses = 16;  // key passes per workgroup (amortises the codebook staging)

__global__ __launch_bounds__(kScanThreads) void k_encode_scan(const EncodeParams p) {
    extern __shared__ __align__(16) float smem[];
    const ssq_encode_args& a = p.a;
    const SsqKeyMap km(a, p.fold);
    const int kv = km.kv;
    const int blk0 = blockIdx.z * p.nbc;
    const int nbc = min(p.nbc, a.n_blocks - blk0);
    const int bd = a.block_dim, nc = a.n_centroids;
    float* cb = smem;                        // [nbc][nc][bd]
    float* cn = cb + (size_t)nbc * nc * bd;  // [nbc][nc]
    const float* cent = a.cent + (int64_t)kv * a.cent_sh + (int64_t)blk0 * nc * bd;
    const float* met = a.metric ? a.metric + (int64_t)kv * a.metric_sh : nullptr;
    const int D = a.head_dim;
    if (met) {  // codebook in the metric space: c' = E_b c, one codeword per thread
        for (int e = threadIdx.x; e < nbc * nc; e += kScanThreads) {
            const int blk = blk0 + e / nc;
            const float* eb = met + (int64_t)blk * bd * D + blk * bd;
            float c[16];
            for (int d = 0; d < bd; ++d) c[d] = cent[(size_t)e * bd + d];
            for (int k = 0; k < bd; ++k) cb[(size_t)e * bd + k] = metric_row(eb + (int64_t)k * D, c, bd);
        }
    } else {
        for (int e = threadIdx.x; e < nbc * nc * bd; e += kScanThreads) cb[e] = cent[e];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nbc * nc; e += kScanThreads) cn[e] = sq_norm(cb + (size_t)e * bd, bd);
    __syncthreads();

    const int64_t* perm = a.perm + (int64_t)kv * a.perm_sh;
    const int keys_per_pass = kScanThreads / nbc;
    const int kk = threadIdx.x / nbc, bl = threadIdx.x - kk * nbc;
    if (kk >= keys_per_pass) return;
    const int blk = blk0 + bl;
    const bool heavy = ssq_is_heavy(a.heavy_mask[0], a.heavy_mask[1], blk);
    const float* cbb = cb + (size_t)bl * nc * bd;
    const float* cnb = cn + (size_t)bl * nc;
    for (int pass = 0; pass < p.passes; ++pass) {
        const int i = (blockIdx.x * p.passes + pass) * keys_per_pass + kk;
        if (i >= km.n_keys) return;
        int b, s;
        km.bs(a, i, b, s);
        const int64_t kbase = (int64_t)b * a.k_sb + (int64_t)kv * a.k_sh + (int64_t)s * a.k_ss;
        float x[16];
        for (int d = 0; d < bd; ++d) x[d] = ssq_load_elem(a.keys, a.k_dtype, kbase + perm[blk * bd + d]);
        int64_t crow, prow;
        out_rows(a, b, kv, s, crow, prow);
        if (heavy) {
            a.codes[crow + blk] = 0;
            const int slot = a.pt_dense ? blk : heavy_ordinal(a.heavy_mask[0], a.heavy_mask[1], blk);
            for (int d = 0; d < bd; ++d) ssq_store_elem(a.pt, a.pt_dtype, prow + (int64_t)slot * bd + d, x[d]);
            continue;
        }
        if (met) {
            const float* eb = met + (int64_t)blk * bd * D + blk * bd;
            float y[16];
            for (int k = 0; k < bd; ++k) y[k] = metric_row(eb + (int64_t)k * D, x, bd);
            for (int k = 0; k < bd; ++k) x[k] = y[k];
        }
        const float xn = sq_norm(x, bd);
        const bool direct = a.direct_dist != 0;
        // pass 1: smallest clamped pre-sqrt value max(e, 0) (first index).  A NaN value (a key
        // with a non-finite element or one whose norm overflows) clamps to 0 as in the
        // reference's sqrt(clamp_min(., 0)) followed by its first argmin of a row holding NaN.
        float emin = INFINITY;
        int jm = 0;
        for (int j = 0; j < nc; ++j) {
            const float e = direct ? direct_dist2(x, cbb + j * bd, bd) : mm_dist2(x, xn, cbb + j * bd, cnb[j], bd);
            const float ec = e > 0.f ? e : 0.f;
            if (ec < emin) { emin = ec; jm = j; }
        }
        // pass 2: the first index whose sqrt equals the minimum's (sqrt merges values at most
        // ~2^-22 apart relatively; indices above jm cannot win).  thr bounds that interval.
        const float fstar = dist_of(emin);
        const float thr = emin > 0.f ? emin * (1.0f + 0x1.0p-20f) : 0.f;
        int best = jm;
        for (int j = 0; j < jm; ++j) {
            const float e = direct ? direct_dist2(x, cbb + j * bd, bd) : mm_dist2(x, xn, cbb + j * bd, cnb[j], bd);
            if (e <= thr && dist_of(e) == fstar) { best = j; break; }
        }
        a.codes[crow + blk] = (uint8_t)best;
    }
}

constexpr size_t kMaxSmem = 160 * 1024;


}  // namespace

extern "C" int ssq_encode(const ssq_encode_args* a, void* stream) {
    if (!a) return ssq_fail(SSQ_ERR_INVALID, "args is NULL");
    if (a->struct_size != sizeof(ssq_encode_args))
        return ssq_fail(SSQ_ERR_ABI, "ssq_encode_args size %u != library's %zu", a->struct_size, sizeof(ssq_encode_args));
    SSQ_REQUIRE(a->keys && a->perm && a->cent && a->codes, "keys, perm, cent and codes must be non-NULL");
    SSQ_REQUIRE(a->batch >= 0 && a->num_kv_heads >= 1 && a->seq_len >= 0, "bad batch/heads/seq_len");
    SSQ_REQUIRE(a->k_dtype >= SSQ_F32 && a->k_dtype <= SSQ_F16, "bad k_dtype");
    SSQ_REQUIRE(a->block_dim >= 1 && a->block_dim <= 16 && a->head_dim % a->block_dim == 0,
                "head_dim must be divisible by block_dim (block_dim <= 16)");
    SSQ_REQUIRE(a->n_blocks == a->head_dim / a->block_dim && a->n_blocks <= 128, "bad n_blocks");
    SSQ_REQUIRE(a->n_centroids >= 1 && a->n_centroids <= kMaxCentroids, "n_centroids must be in [1, %d]", kMaxCentroids);
    const bool any_heavy = a->heavy_mask[0] || a->heavy_mask[1];
    SSQ_REQUIRE(!any_heavy || a->pt, "heavy blocks need a passthrough output");
    if (any_heavy) SSQ_REQUIRE(a->pt_dtype >= SSQ_F32 && a->pt_dtype <= SSQ_F16, "bad pt_dtype");
    if (a->slot_mapping) SSQ_REQUIRE(a->page_size >= 1, "paged output needs page_size >= 1");
    SSQ_REQUIRE(a->direct_dist == 0 || a->direct_dist == 1, "direct_dist must be 0 or 1");
    if (a->batch == 0 || a->seq_len == 0) return SSQ_OK;
    hipStream_t st = (hipStream_t)stream;
    // the direct distance (a cdist over at most 25 x 25 rows) runs on the exact scan only: the MFMA
    // screen and the grid search certify candidates against the mm formulation's rounding
    SSQ_UNSUPPORTED(!a->direct_dist || a->kernel == 0 || a->kernel == 1,
                    "direct_dist runs on the exact scan (kernel 0 or 1), not kernel %d", a->kernel);
    if (a->n_centroids > 256) {  // 16- / 32-bit codes
        SSQ_UNSUPPORTED(a->kernel == 0 || a->kernel == 1,
                        "n_centroids=%d encodes under kernel 0, or 1 for the exact scan, not kernel %d", a->n_centroids,
                        a->kernel);
        const int cw = ssq_code_width(a->n_centroids);
        SSQ_REQUIRE((uintptr_t)a->codes % cw == 0, "%d-bit codes must be %d-byte aligned", 8 * cw, cw);
        // The screen stages every codebook once per 512 keys of a KV head and folds its groups, which for few
        // keys, and up to about 2^24 (key, block, codeword) triples, costs more than the exact scan split
        // over lanes: bf16 keys of head_dim 128, 8 heads, 8 rows each at 4,096 codewords of dim 4 (2^23)
        // 18 us on the scan and 34 on the screen, at 65,535 (2^27) 215 and 454.  Codebooks of dims 1 and 2
        // stay on the scan: many codewords then lie within the screen's bound of the nearest, which leaves
        // most pairs to a scan of its own (2,048 keys at 1,024 codewords of dim 1: 303 us on the scan, 612
        // on the screen; 4,096 at 1,024 of dim 2, 323 and 136 when centred, 590 with an offset of 30 standard
        // deviations).  The codes are the same.
        const int64_t keys = (int64_t)a->batch * a->seq_len;
        const int64_t work = keys * a->num_kv_heads * a->n_blocks * a->n_centroids;
        if (a->kernel == 0 && !a->direct_dist && a->block_dim >= 3 && a->block_dim <= 8 && keys >= 32 &&
            work > (int64_t)1 << 24)
            return ssq_encode_tile_run(a, st);
        return ssq_encode_wide_run(a, st);
    }
    if (!a->direct_dist && (a->kernel == 3 || (a->kernel == 0 && a->grid && ssq_encode_grid_supported(a))))
        return ssq_encode_grid_run(a, st);
    const bool tile_ok = a->n_centroids == 256 && a->block_dim <= 10 && !a->direct_dist;
    const int kernel = a->kernel == 0 ? (tile_ok ? 2 : 1) : a->kernel;
    if (kernel == 2) {
        SSQ_UNSUPPORTED(tile_ok, "MFMA encode needs n_centroids == 256 and block_dim <= 10");
        return ssq_encode_tile_run(a, st);
    }
    EncodeParams p;
    p.a = *a;
    // exact scan
    int nbc = a->n_blocks < kScanThreads ? a->n_blocks : kScanThreads;
    while (nbc > 1 && (size_t)nbc * a->n_centroids * (a->block_dim + 1) * 4 > 96 * 1024) --nbc;
    p.nbc = nbc;
    // folded (short sequences): one pass per workgroup, so the few keys spread over workgroups
    p.fold = ssq_encode_fold(a, (kScanThreads / nbc) * kScanPasses);
    p.passes = p.fold ? 1 : kScanPasses;
    const int keys_per_wg = (kScanThreads / nbc) * p.passes;
    const int64_t n_keys = p.fold ? (int64_t)a->batch * a->seq_len : a->seq_len;
    dim3 grid((unsigned)((n_keys + keys_per_wg - 1) / keys_per_wg), p.fold ? a->num_kv_heads : a->batch * a->num_kv_heads,
              (a->n_blocks + nbc - 1) / nbc);
    const size_t smem = (size_t)nbc * a->n_centroids * (a->block_dim + 1) * 4;
    int rc = ssq_allow_lds((const void*)k_encode_scan, (int)kMaxSmem, "hipFuncSetAttribute(encode)");
    if (rc) return rc;
    hipLaunchKernelGGL(k_encode_scan, grid, dim3(kScanThreads), smem, st, p);
    return ssq_check_hip(hipGetLastError(), "k_encode_scan launch");
}
