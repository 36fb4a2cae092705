// Host arithmetic of the C ABI's calls: the byte sizes of token arrays, the layout of a
// call's workspace regions, how long batches are cut into launches, and the rules that choose
// a kernel by sizes alone.  It is kept apart
// from nnq_abi.cpp (which makes the HIP runtime calls) so that the sanitizer harness
// (tests/sanitize) runs the same code on the CPU over ragged and extreme shapes.
#include <algorithm>
#include <cmath>

#include "nnq_internal.h"

namespace nnq {

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

bool array_bytes(int64_t rows, int64_t cols, size_t elem, size_t *out) {
    *out = 0;
    if (rows < 0 || cols < 0) return false;
    size_t a = 0;
    if (__builtin_mul_overflow((size_t)rows, (size_t)cols, &a)) return false;
    return !__builtin_mul_overflow(a, elem, out);
}

bool plan_regions(const size_t *sizes, int n, size_t *offsets, size_t *total) {
    size_t at = 0;
    for (int i = 0; i < n; i++) {
        offsets[i] = at;
        if (sizes[i] == 0) continue;  // an absent region takes no space
        // the next region starts at the 256-byte boundary after this one
        size_t end = 0;
        if (__builtin_add_overflow(at, sizes[i], &end) || end > SIZE_MAX - 255) return false;
        at = align256(end);
    }
    *total = at;
    return true;
}

int64_t moe_chunk_tokens(int64_t tokens, int top_k) {
    if (tokens <= 0 || top_k <= 0) return 0;
    return std::max<int64_t>(1, std::min<int64_t>(tokens, kMoeChunkAssign / top_k));
}

int64_t gemm_chunk_rows(int64_t m, int64_t k) {
    if (m <= 0 || k <= 0) return 0;
    // the GEMMs address an activation plane (and its f32 hi + lo pair) with 32-bit byte
    // offsets: 2 planes * rows * K * 2 bytes stays below 2^31
    const int64_t lim = ((int64_t)1 << 31) - 1;
    int64_t rows = lim / (4 * k);
    if (rows >= 256) rows = rows / 256 * 256;  // whole 256-row tiles per launch
    return std::min(m, std::max<int64_t>(1, rows));
}

// ---- dispatch rules ----------------------------------------------------------------

// The path of a linear call of m tokens, by measured crossovers on MI355X (us, x f32 / bf16):
//  - 1 and 2 tokens: one decode-GEMV pass;
//  - 3 to 16: the few-row GEMM (nnq_gemm_few.hip) from 5 tokens on (Q8_0 4096x4096, 12 tokens:
//    14.3 / 17.0 as passes / GEMM, 12.8 / 7.5 there; Q6_K 12288x4096, 8 tokens: 26.8 / 26.3 as
//    two passes, 14.0 / 12.1).  Below that a GEMV pass of 4 tokens has the shorter prologue
//    (Q6_K 4096x4096: 6.2 against 8.4 / 7.4), except over eight tiles per CU or more (3 f32 tokens,
//    pass against few rows: Q6_K 151936 x 4096 133 / 97, 40960 x 2048 19.9 / 17.6; Q8_0 40960 x 2048
//    19.0 / 16.8; Q4_K 40960 x 4096 29.2 / 24.5; under 2048 k the pass is faster, 40960 x 1024
//    11.3 / 12.1, 10.8 / 11.3 and 8.7 / 11.4, but its sums are the less exact ones, so that the
//    rule has no line there).  Q4_K with f32 x takes it from 7
//    tokens (4096x4096: 5 and 6 as two passes 8.6 and 9.0 against 9.1 and 9.3; 8: 10.5 against
//    9.6), from 5 with two tiles per CU (24576 rows: 30.0 against 19.3) or K over 8192 (6
//    tokens at 4096x12288: 19.0 against 17.2).  Q4_K with bf16 x keeps the thin GEMM, which
//    stages nothing, up to that many tiles (16 tokens: 12288x4096 10.0 against 13.0, 24576
//    rows 18.8 against 19.5, 60000 rows 45.2 against 37.6).  Over 8 tokens of Q6_K are two
//    launches there: four tiles per CU of one or two units leave them to the MFMA GEMM (16 bf16
//    tokens, GEMM against few rows: 65536 x 256 14.4 / 25.4, x 512 20.7 / 26.5, x 1024 33.9 / 29.4;
//    8192 x 512 13.7 / 11.3);
//  - other counts: the MFMA GEMM.
// 1 where the few-row GEMM takes the call.
int nnq_rule_few_rows(int fmt, int64_t ntile, int64_t k, int64_t m, int x_bf16) {
    if (m < 3 || m > 16 || k > ((int64_t)1 << 24) || ntile >= ((int64_t)1 << 31)) return 0;
    if (fmt == NNQ_FMT_Q6_K && m > 8 && ntile >= 1024 && k <= 512) return 0;
    if (ntile >= 2048) return 1;  // eight tiles per CU
    if (fmt != NNQ_FMT_Q4_K) return m > 4;
    if (x_bf16) return 0;
    return m > 6 || (m > 4 && (ntile >= 512 || k > 8192));
}

// Shapes the Q4_K ring kernel takes (N % 128 == 0; f32 activations run their staged hi and lo
// planes as two halves of the work, summed by the finalize):
// BM x BN tiles, BM the smallest of 32, 64, 128 holding M (128 beyond), BN 192 or 128
// (dividing N), K split 1, 2, 4, 8 or 16 ways (a divisor of the super-block count leaving
// at least 4 super-blocks per workgroup, 2 with BM < 128).  Of these, the plan with the
// least estimated time: rounds of workgroups (one resident per CU: the rings of the small
// row tiles are deepened to 6 stages, which LDS holds once) times stages per workgroup, a 128-wide
// stage at 0.8 of a 192-wide one, plus one stage for the split-K finalize.  (Assuming two
// resident workgroups with shallower rings measured 5-25% slower at M = 16 to 64.)
// Returns the K split, or 0 when the shape does not fit.
int nnq_rule_gemm_ring(int64_t m, int64_t ntile, int64_t nblk, int x_bf16, int *bn, int *bm) {
    if (m < 1 || nblk < 1) return 0;
    const int npl = x_bf16 ? 1 : 2;  // f32 activations: hi and lo planes, each a full pass
    const int rows = m <= 32 ? 32 : (m <= 64 ? 64 : 128);
    const int64_t ncols = ntile * 16, nrt = (m + rows - 1) / rows;
    const int min_sb = rows == 128 ? 4 : 2;
    double best_cost = 0.0;
    int best_bn = 0, best_ks = 0;
    for (int cand : {192, 128}) {
        if (ncols % cand) continue;
        for (int ks = 1; ks <= 16; ks *= 2) {
            if (nblk % ks || (ks > 1 && nblk / ks < min_sb)) continue;
            const int64_t rounds = (nrt * (ncols / cand) * ks * npl + 255) / 256;
            const double cost = (double)rounds * (double)(nblk / ks) * (cand == 192 ? 1.0 : 0.8) + (ks * npl > 1 ? 1.0 : 0.0);
            if (best_bn == 0 || cost < best_cost) {
                best_cost = cost;
                best_bn = cand;
                best_ks = ks;
            }
        }
    }
    if (best_bn == 0) return 0;
    if (bn) *bn = best_bn;
    if (bm) *bm = rows;
    return best_ks;
}

// The wide kernel's shape rules: more than 128 rows (below, half of a 256-row tile or more is
// padding: f32 x, 100 x 4096 x 12288 109 us against the ring's 51), whole 16-row weight tiles
// and a 16-byte aligned output (the epilogue writes 16-byte row chunks), K <= 4096 * 3 (the
// staging keeps the row in one workgroup's registers and its sub-block sums in LDS), and at
// least 128 workgroups.  Column tiles per workgroup (6, 4 or 8) and K split (1 to 8 equal parts
// of whole super-blocks) are the ones with the least estimated time: rounds of workgroups over
// the CUs, each 3 us and its super-blocks times the measured time of one (us, 6, 4 and 8 tiles: bf16 x
// 3.8, 3.0 and 5.0, f32 x 6.2, 5.2 and 7.8: more tiles read each A fragment less often), plus
// the slabs' write, read and launch.  With bf16 x a part of two super-blocks, whose prologue nothing
// hides, counts as 2.7 and each further part adds 1.8% (without the two: 400 x 2560 x 2560 in 8 tiles and
// K in five 27.9 us, in 4 tiles and K in two 25.0; 200 x 6144 x 2048 25.4 and 23.6; 129 x 8192 x 3072 28.7
// and 26.6).
// 512 rows of f32 x take 107 us at 12288 x 4096 (6 tiles; the ring kernel over two planes 153) and
// 115 at 4096 x 12288 (8 tiles, K in four; 4 tiles and K in two 134, ring 155), of bf16 x there 77
// (4 tiles 83); 203 rows of f32 x at 12288 x 4096 take 6 tiles and K in two (256 workgroups).
// With random x these rates are the chip's power limit for f16 products: a library f16 GEMM
// of 512 x 12288 x 4096 takes 58 us (44 with x = 0), this kernel 66 with its staging (60).
// With f32 x the ring kernel keeps what it does faster, above all K of a prime number of super-blocks,
// which cannot be split here (260 x 5376 x 11008 125 us there, 187 here; 384 x 4736 x 1792 34 and 39).
// Both sides' times are estimated with constants fitted to 288 calls of the ring and 713 of this
// kernel, 4% and 5% off in the mean: us, per million of x, per MB of slabs (the ring's two planes have
// one each), per round and per super-block of a round (the ring's 128-column tiles 0.8 of its wide ones).
// h_out: the call is an MLP's gate | up and wants h = silu(gate) * up, which this kernel writes itself
// where K is not split and the ring leaves to a launch of about 4 us (f32 forwards, ring / wide gate | up: 260
// tokens of 768 x 2048 49.5 / 44.4 us, 129 of 1792 x 4608 66.3 / 61.7; 129 of 2816 x 4096 72.0 / 78.8).
// Returns the column tiles per workgroup (0: the ring kernel takes the shape) and the K split.
int nnq_rule_gemm_wide(int64_t m, int64_t ntile, int64_t nblk, int x_bf16, int h_out, int *ks) {
    if (m <= 128 || nblk > 48) return 0;
    const int64_t nrt = (m + 255) / 256, n = ntile * 16;
    const int tiles[3] = {6, 4, 8};
    const float sb_us[2][3] = {{3.8f, 3.0f, 5.0f}, {6.2f, 5.2f, 7.8f}};
    const float y_mb = (float)(m * n) * 4.0e-6f;
    float best = 0.0f;
    int at = -1, best_ks = 0;
    for (int i = 0; i < 3; i++) {
        if (ntile % tiles[i]) continue;
        for (int split = 1; split <= 8; split++) {
            const int64_t wg = nrt * (ntile / tiles[i]) * split;
            if (wg < 128 || nblk % split || nblk / split < 2) continue;
            const float sb = x_bf16 ? std::max((float)(nblk / split), 2.7f) : (float)(nblk / split);
            float us = (float)((wg + 255) / 256) * (3.0f + sb * sb_us[x_bf16 ? 0 : 1][i]);
            if (split > 1) us += 3.0f + (float)(split + 1) * y_mb * 0.25f;
            if (x_bf16) us *= 1.0f + 0.018f * (float)(split - 1);
            if (at < 0 || us < best) {
                best = us;
                at = i;
                best_ks = split;
            }
        }
    }
    if (at < 0) return 0;
    int bn = 0;
    const int rks = x_bf16 ? 0 : nnq_rule_gemm_ring(m, ntile, nblk, 0, &bn, nullptr);
    if (rks) {
        const float x_m = (float)m * (float)(nblk * 256) * 1.0e-6f, f32_us[3] = {4.7f, 3.9f, 5.8f};
        const int64_t rounds = (nrt * (ntile / tiles[at]) * best_ks + 255) / 256;
        const int64_t rrounds = ((m + 127) / 128 * (n / bn) * rks * 2 + 255) / 256;
        const float slabs = best_ks > 1 ? 0.5f + 0.22f * (float)(best_ks + 1) * y_mb : 0.0f;
        const float wide = 7.1f + 1.37f * x_m + (float)rounds * (3.8f + (float)(nblk / best_ks) * f32_us[at]) + slabs;
        const float ring = 10.4f + 1.05f * x_m + 0.34f * (float)(2 * rks + 1) * y_mb +
                           3.15f * (float)(rrounds * (nblk / rks)) * (bn == 192 ? 1.0f : 0.8f);
        if (ring + (h_out && best_ks == 1 ? 4.0f : 0.0f) < wide) return 0;
    }
    if (ks) *ks = best_ks;
    return tiles[at];
}

// The wide Q6_K kernel's shape rules: bf16 activations, more than 128 rows, whole groups of 8 weight tiles, K up
// to 4096 * 3 (the activation staging), a 16-byte aligned output, and at least 192 workgroups, or
// 128 with 8 super-blocks each.  The K split (1 to 8 equal parts of two or more super-blocks) is
// the one with the least estimated time: rounds of workgroups over the CUs, each 3 us and 7.8 us
// per super-block, plus the slabs; where that is not below the block kernel's estimate, that
// kernel keeps the shape (1000 x 2048 x 2560: 57 us wide, 49 there; 274 x 19200 x 7168, whose
// second row tile is nearly all padding: 285 and 277).  A second 128-row tile of up to 32 rows
// costs the block kernel less than a full one, 12% in its estimate (256, 160 and 129 x 40960 x
// 1024: 88, 62 and 59 us, wide 69, 67 and 66; 129 x 9728 x 2560: 45.7, wide 47.9).  Measured (block kernel -> wide): 512 x
// 4096 x 12288 134 -> 105 us, 512 x 12288 x 4096 167 -> 123, 300 x 4096 x 4096 67 -> 49, 200 x
// 4096 x 12288 108 -> 66, 256 x 24576 x 1024 61 -> 42.
// Returns the K split (0: the block kernel takes the shape).
int nnq_rule_gemm_wide6(int64_t m, int64_t ntile, int64_t nblk) {
    if (m <= 128 || nblk > 48 || ntile % 8) return 0;
    const int64_t base = (m + 255) / 256 * (ntile / 8), n = ntile * 16;
    // the block kernel: 128-row tiles at about 350 TFLOP/s, its staging and slab sum 12 us
    float best = 12.0f + 2.0f * (float)((m + 127) / 128 * 128) * (float)n * (float)(nblk * 256) / 350.0e6f;
    if (m <= 160) best *= 0.88f;
    int ks = 0;
    for (int split = 1; split <= 8; split++) {
        const int64_t wg = base * split;
        if (nblk % split || wg < 128 || nblk / split < 2 || (wg < 192 && nblk / split < 8)) continue;
        const float slabs = split > 1 ? 3.0f + (float)(split + 1) * (float)(m * n) * 4.0f / 4.0e6f : 0.0f;
        const float us = (float)((wg + 255) / 256) * (3.0f + (float)(nblk / split) * 7.8f) + slabs;
        if (us < best) {
            best = us;
            ks = split;
        }
    }
    return ks;
}

// Whether a MoE layer's experts run as moe_few_kernel's items (up to kMoeFewT tokens and
// kMoeFewAssign assignments) rather than as moe_stream_kernel's workgroups.  The items' time grows
// with the passes of four rows over an expert's weights, expected here for even routing; the
// streams' hardly does (a pass of theirs is 64 rows), so there is a number of passes where they
// cross: 28 with bf16 x and 22.5 with f32 x (which the items split on each pass, the streams
// once) for 2880 x 2880 experts, 5 and 4.5 more with each halving of an expert (an item of a small
// one is mostly its fixed part).  Streams of over 32 experts are more workgroups than CUs, and over
// 96 column streams take a wave more than one each: both raise it.  Measured (us, streams / items,
// top 8): 32 experts of 2880 x 2880, 6 bf16 tokens 104 / 99, 12 108 / 123, 16 109 / 151, 4 f32 tokens
// 127 / 127, 16 132 / 238; 16 such experts, 10 bf16 tokens 100 / 96, 16 101 / 126; 32 of 2048 x 2048, 12
// bf16 tokens 94 / 90, 16 94 / 109; 64 of 1024 x 768, 16 f32 tokens 79 / 71.
int nnq_rule_moe_few(int64_t experts, int64_t hidden, int64_t inter, int64_t tokens, int top_k, int x_bf16) {
    if (tokens > kMoeFewT || tokens * top_k > kMoeFewAssign) return 0;
    // an expert's rows are binomial: P(n) from P(n - 1)
    const double p = (double)top_k / (double)experts;
    double passes = (double)((tokens + 3) / 4);
    if (p < 1.0) {
        double pn = std::pow(1.0 - p, (double)tokens);
        passes = 0.0;
        for (int64_t n = 1; n <= tokens; n++) {
            pn *= (double)(tokens - n + 1) / (double)n * p / (1.0 - p);
            passes += pn * (double)((n + 3) / 4);
        }
    }
    passes *= (double)experts;
    const double halvings = std::max(0.0, std::log2(2880.0 * 2880.0 / ((double)hidden * (double)inter)));
    const double cross = x_bf16 ? 28.0 + 5.0 * halvings : 22.5 + 4.5 * halvings;
    const int64_t sets = (experts + 31) / 32, rounds = (inter / 32 + 95) / 96 + (hidden / 32 + 95) / 96;
    return passes <= cross * (1.0 + 1.25 * (double)(sets - 1)) * 0.5 * (double)rounds;
}

}  // namespace nnq
