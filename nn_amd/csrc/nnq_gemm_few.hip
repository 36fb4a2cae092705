// GEMM over a few token rows on gfx950, Y[m, n] = X[m, k] . W[n, k]^T (+ bias), in one launch
// that reads the weight once: Q8_0 and Q4_K weights for up to 16 rows of f32 or bf16 x, Q6_K
// for up to 8 (quantized_linear over a served batch, crates/nn-core/src/dyn_tensor/
// quantized_matmul.rs:367-406); 9 to 16 rows of Q6_K are two launches, which read the weight
// twice.  The weight is the decode GEMVs' tile16 image.
//
// Bound: the weight stream from HBM (an LM head of 151936 x 4096 in Q6_K: 511 MB, 73 us), and
// close behind it the VALU that forms the MFMA's B operands and applies the block scales, so
// everything else is kept out of the loop over tiles:
//  * One workgroup per CU takes a contiguous run of 16-column weight tiles and up to 16 units
//    of 256 k; a longer K is split over workgroups (f32 slabs summed by few_sum_kernel), so
//    that a wave owns ONE unit: its activation is converted once into MFMA A operands held in
//    registers and multiplied with the unit's codes of all the workgroup's tiles.  With 8 or
//    fewer units the waves form 2 or 4 groups that take the tiles in turn.
//  * The raw bytes of the wave's next tile are in flight while the current one is computed.
//  * The waves' sums of a round of tiles meet in LDS: one barrier per round, the buffers of
//    two rounds alternating.
//
// Arithmetic: x of a (row, unit) is scaled by a power of two (its largest magnitude into
// [2^14, 2^15)) to f16 (bf16 x) or an f16 hi + lo pair (f32 x, ~22 bits); codes become exact
// normal f16 integers (0x6400 | c is 1024 + c; one packed add takes 1024 and the format's
// offset off), so every product is exact in f32.  The decode GEMVs' form, codes as f16
// subnormals, saves that add but loses precision where it counts: the matrix core aligns the
// products of an instruction by their operands' exponent fields, so a subnormal code costs the
// sum up to 10 bits (f32 x, Q6_K, K = 2304: error against 64 bits 1.1e-5 with subnormal codes
// and the offset from an MFMA with a constant, 2e-7 here).  The lo product comes first: added
// to a finished hi sum its low bits would be cut off one instruction at a time.
// Measured (us, before -> now; before: GEMV passes or the prefill GEMM, each of which reads the
// weight or stages the activation more than once): Q6_K LM head 151936 x 4096, 8 bf16 rows 260
// -> 97, 16 rows 271 -> 204 (two launches); Q8_0 4096 x 4096, 12 bf16 rows 17.3 -> 7.8;
// Q4_K 4096 x 12288, 6 f32 rows 18.3 -> 16.0 (K split three ways), 12288 x 4096, 16 f32 rows
// 27.3 -> 18.0.
// Registers: 16 waves leave 128 each, which the f32 plane form (9 to 16 rows) passes by 6 (Q4_K)
// and 10 (Q8_0), spilled; the other forms fit.
// Rows: Q8_0 and Q4_K have one scale per 32 k, one MFMA row per token.  A Q6_K scale covers 16 k,
// so token t takes rows 2t and 2t + 1, each with zeros in the other sub-block's half of k.
// A NaN or infinity in a token's unit makes that token's outputs NaN.
#include <algorithm>

#include "nnq_device.h"
#include "nnq_internal.h"

namespace nnq {

namespace {

constexpr int kFewWaves = 16;
constexpr int kFewRB = 4;  // tiles per round

struct FewArgs {
    const uint8_t *qs, *hdr;
    const void *x;
    const float *bias;
    void *y;     // [m][n], or with ks > 1 f32 slabs [ks][m][n] without the bias
    int y_bf16;
    int m, units, ntile;
    int ks;      // workgroups that share a tile's K
    int up;      // units of a workgroup (at most 16) rounded up to 4, 8 or 16: 16 / up wave groups
    int64_t k, n;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t few_rsrc(const void *p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)min(bytes, (int64_t)0x7FFFFFF0), 0x00020000);
}
// AUX 2: non-temporal (the weight stream, read once), 0: default
template <int AUX>
__device__ __forceinline__ u32x4 few_load4(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, AUX));
}

// f16(a * s) | f16(b * s) << 16, and the f16 residuals a * s - hi.x, b * s - hi.y (each formed
// exactly by the FMA)
__device__ __forceinline__ uint32_t few_hi2(float a, float b, float s) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0\n\tv_fma_mixhi_f16 %0, %3, %2, 0" : "=&v"(r) : "v"(a), "v"(s), "v"(b));
    return r;
}
__device__ __forceinline__ uint32_t few_lo2(float a, float b, float s, uint32_t hi) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, %2, -%4 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, %3, %2, -%4 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(r)
        : "v"(a), "v"(s), "v"(b), "v"(hi));
    return r;
}
__device__ __forceinline__ float few_absmax(float m, float a, float b) {
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint32_t few_umax_rows(uint32_t v) {  // over the four 16-lane groups
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = max(a[0], a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return max(b[0], b[1]);
}

// per format: the raw bytes of one (tile, unit), their loads, and the products of one unit
template <int FMT>
struct FewRaw;
template <>
struct FewRaw<NNQ_FMT_Q4_K> {
    u32x2 q[4];
    u32x4 h;
};
template <>
struct FewRaw<NNQ_FMT_Q8_0> {
    u32x4 q[4];
    u32x4 h;
};
template <>
struct FewRaw<NNQ_FMT_Q6_K> {
    u32x3 q[4];
    u32x4 s;
    uint32_t d;
};

template <int FMT>
constexpr int few_qbytes() { return FMT == NNQ_FMT_Q4_K ? 2048 : FMT == NNQ_FMT_Q8_0 ? 4096 : 3072; }
template <int FMT>
constexpr int few_hbytes() { return FMT == NNQ_FMT_Q6_K ? 288 : 256; }

template <int FMT>
__device__ __forceinline__ void few_load(const FewArgs &a, int tile, int u, int lane, FewRaw<FMT> &w) {
    const size_t base = (size_t)tile * a.units;
    const __amdgpu_buffer_rsrc_t rq = few_rsrc(a.qs + base * few_qbytes<FMT>(), (int64_t)a.units * few_qbytes<FMT>());
    const __amdgpu_buffer_rsrc_t rh = few_rsrc(a.hdr + base * few_hbytes<FMT>(), (int64_t)a.units * few_hbytes<FMT>());
    const int G = lane >> 4, c16 = lane & 15;
    const int qo = u * few_qbytes<FMT>(), ho = u * few_hbytes<FMT>();
    if constexpr (FMT == NNQ_FMT_Q4_K) {
        // lane (G, c) of group p takes bytes 8G .. 8G + 7 of row c's group p: low nibbles
        // sub-block 2p, high 2p + 1
        w.h = few_load4<2>(rh, 16 * c16, ho);
#pragma unroll
        for (int p = 0; p < 4; p++)
            w.q[p] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(
                                                   rq, (G >> 1) * 1024 + c16 * 16 + 8 * (G & 1), qo + 256 * p, 2));
    } else if constexpr (FMT == NNQ_FMT_Q8_0) {
        w.h = few_load4<2>(rh, 16 * c16, ho);
#pragma unroll
        for (int p = 0; p < 4; p++) w.q[p] = few_load4<2>(rq, 16 * lane, qo + 1024 * p);
    } else {
        w.s = few_load4<2>(rh, 16 * c16, ho);
        w.d = __builtin_amdgcn_raw_buffer_load_b16(rh, 256 + 2 * c16, ho, 2);
#pragma unroll
        for (int p = 0; p < 4; p++)
            w.q[p] = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(rq, 12 * lane, qo + 768 * p, 2));
    }
}

// XM, the activation: bf16, f32 as hi and lo operands of the same rows, or (up to 8 tokens of
// Q8_0 and Q4_K) f32 with the hi and lo parts of token t in rows 2t and 2t + 1 of one operand
enum { kFewBf16 = 0, kFewPlanes = 1, kFewPairs = 2 };

// FMT: weight format.  Lane 16G + c16: A row c16 (elements
// 8G .. 8G + 7 of a 32-k step), B and D column c16 (row c16 of the tile), D rows 4G .. 4G + 3.
template <int FMT, int XM>
__global__ __launch_bounds__(kFewWaves * 64) void gemm_few_kernel(FewArgs a) {
    constexpr bool Q6 = FMT == NNQ_FMT_Q6_K, XB = XM == kFewBf16, PAIR = XM == kFewPairs;
    constexpr bool TWO = Q6 || PAIR;              // two rows per token
    constexpr int NP = XM == kFewPlanes ? 2 : 1;  // operands per step
    constexpr int NE = TWO ? 2 : 4;               // outputs of a lane (TWO: tokens 2G, 2G + 1)
    static_assert(!(Q6 && PAIR), "a Q6_K token's rows are its sub-blocks");
    constexpr int RB = kFewRB;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ float btab[kFewWaves][16];
    __shared__ __attribute__((aligned(16))) float stab[FMT == NNQ_FMT_Q4_K ? kFewWaves : 1][16][8];
    float *red = reinterpret_cast<float *>(smem);  // [2][wave][tile of the round][NE][lane]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = lane >> 4, c16 = lane & 15;
    const int k = (int)a.k;
    // K part and tile run of the workgroup; unit and tile group of the wave
    const int part = (int)blockIdx.x % a.ks, run = (int)blockIdx.x / a.ks, runs = (int)gridDim.x / a.ks;
    const int t_lo = (int)((int64_t)run * a.ntile / runs), t_hi = (int)((int64_t)(run + 1) * a.ntile / runs);
    const int u_lo = part * a.units / a.ks, nu = (part + 1) * a.units / a.ks - u_lo;  // <= up
    const int ng = kFewWaves / a.up, grp = wv / a.up, u = u_lo + wv % a.up;

    // activation: row c16's token (rows past m read zeros past the range), for Q6_K only the
    // row's half of each 32 k
    const int tok = TWO ? c16 >> 1 : c16;
    const bool live = tok < a.m && (!Q6 || (G >> 1) == (c16 & 1));
    constexpr int xe = XB ? 2 : 4;
    const __amdgpu_buffer_rsrc_t rx = few_rsrc(a.x, (int64_t)a.m * k * xe);
    const uint32_t xoff = live ? (uint32_t)((tok * k + 8 * G) * xe) : 0x80000000u;
    u32x4 A[NP][8];
    u32x4 As;  // Q4_K: the sub-blocks' sums of x as f16 hi and lo, the operand of the min term
    float back[NE];
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    auto prod = [&](int s, u32x4 b, floatx4 c) {
        if constexpr (NP == 2) c = mfma16x16x32_f16(A[NP - 1][s], b, c);
        return mfma16x16x32_f16(A[0][s], b, c);
    };
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    struct XRaw {
        u32x4 v[8 * (XB ? 1 : 2)];
    };
    auto x_load = [&](int u, XRaw &x) {
        // (Q8_0's last unit may be partial: steps past k read zeros)
        auto &v = x.v;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int e = u * 256 + 32 * s;
            const uint32_t off = FMT != NNQ_FMT_Q8_0 || e < k ? xoff : 0x80000000u;
            if constexpr (XB) {
                v[s] = few_load4<0>(rx, (int)off, e * 2);
            } else {
                v[2 * s] = few_load4<0>(rx, (int)off, e * 4);
                v[2 * s + 1] = few_load4<0>(rx, (int)(off + 16), e * 4);
            }
        }
    };
    auto x_stage = [&](const XRaw &x) {
        const auto &v = x.v;
        uint32_t mb;
        if constexpr (XB) {
            typedef uint16_t us2 __attribute__((ext_vector_type(2)));
            us2 mx = {0, 0};
#pragma unroll
            for (int s = 0; s < 8; s++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    mx = __builtin_elementwise_max(mx, __builtin_bit_cast(us2, v[s][i] & 0x7FFF7FFFu));
            const uint32_t w = __builtin_bit_cast(uint32_t, mx);
            mb = max(w & 0xFFFF0000u, w << 16);
        } else {
            float mx = 0.0f;  // (drops NaN elements: each stays NaN in its own operand)
#pragma unroll
            for (int s = 0; s < 16; s++)
#pragma unroll
                for (int i = 0; i < 4; i += 2)
                    mx = few_absmax(mx, __uint_as_float(v[s][i]), __uint_as_float(v[s][i + 1]));
            mb = __float_as_uint(mx);
        }
        mb = few_umax_rows(mb);
        if constexpr (Q6) mb = max(mb,  // the token's other row holds its other halves
                                    (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mb, 0xB1, 0xF, 0xF, true));
        float s, bk;
        f16_prescale(__uint_as_float(mb), s, bk);
#pragma unroll
        for (int q = 0; q < 8; q++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float f0, f1;
                if constexpr (XB) {
                    f0 = __uint_as_float(v[q][i] << 16);
                    f1 = __uint_as_float(v[q][i] & 0xFFFF0000u);
                } else {
                    f0 = __uint_as_float(v[2 * q + (i >> 1)][2 * (i & 1)]);
                    f1 = __uint_as_float(v[2 * q + (i >> 1)][2 * (i & 1) + 1]);
                }
                const uint32_t hi = few_hi2(f0, f1, s);
                if constexpr (PAIR) {
                    const uint32_t lo = few_lo2(f0, f1, s, hi);
                    A[0][q][i] = (c16 & 1) ? lo : hi;
                } else {
                    A[0][q][i] = hi;
                    if constexpr (NP == 2) A[NP - 1][q][i] = few_lo2(f0, f1, s, hi);
                }
            }
            if constexpr (!XB) __builtin_amdgcn_sched_barrier(0);  // raw x dies as operands are born
        }
        // 2^-s of the D rows' tokens, through the wave's table
        if (G == 0 && (!TWO || !(c16 & 1))) btab[wv][tok] = bk;
        if constexpr (FMT == NNQ_FMT_Q4_K) {
            // sums of the scaled x over each sub-block (every column of the product with ones):
            // column s's lanes keep step s's
            const u32x4 ones = {0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};  // f16 1.0
            floatx4 mine = zero;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const floatx4 S = prod(q, ones, zero);
                if (c16 == q) mine = S;
            }
            if (c16 < 8) {
#pragma unroll
                for (int e = 0; e < NE; e++) stab[wv][NE * G + e][c16] = PAIR ? mine[2 * e] + mine[2 * e + 1] : mine[e];
            }
        }
        wave_sync();
#pragma unroll
        for (int e = 0; e < NE; e++) back[e] = btab[wv][NE * G + e];
        if constexpr (FMT == NNQ_FMT_Q4_K) {
            // k slots 0 .. 7 (lane group 0): the hi parts of 2^-8 * sum, in the lo rows of a pair
            // the lo parts; without pairs slots 8 .. 15 (group 1) hold the lo parts
            const floatx4 s0 = *reinterpret_cast<const floatx4 *>(&stab[wv][tok][0]);
            const floatx4 s1 = *reinterpret_cast<const floatx4 *>(&stab[wv][tok][4]);
            const bool lo = PAIR ? (c16 & 1) != 0 : G == 1, any = PAIR ? G == 0 : G < 2;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float f0 = i < 2 ? s0[2 * i] : s1[2 * i - 4], f1 = i < 2 ? s0[2 * i + 1] : s1[2 * i - 3];
                const uint32_t hi = few_hi2(f0, f1, 0x1p-8f), l = few_lo2(f0, f1, 0x1p-8f, hi);
                As[i] = any ? (lo ? l : hi) : 0u;
            }
        }
        wave_sync();
    };
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    // codes c in the low 10 bits of each half of v (the rest masked off by m) -> f16 c - off
    auto code2 = [](uint32_t v, uint32_t m, float off) {
        const h2 k = {(_Float16)(-1024.0f - off), (_Float16)(-1024.0f - off)};
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, (v & m) | 0x64006400u) + k);
    };
    // a token's two rows: one after the other into its sum, scaled by fa and fb
    auto add2 = [](float *T, const floatx4 &P, float fa, float fb) {
#pragma unroll
        for (int t = 0; t < 2; t++) T[t] = __builtin_fmaf(fb, P[2 * t + 1], __builtin_fmaf(fa, P[2 * t], T[t]));
    };
    auto compute = [&](const FewRaw<FMT> &w, float y[NE]) {
        if constexpr (FMT == NNQ_FMT_Q4_K) {
            // d, dmin and the sub-blocks' 6-bit scales and mins (get_scale_min_k4,
            // crates/nn-core/src/layers/quantized/linear.rs:166-176)
            const uint32_t sc[2] = {w.h[1] & 0x3F3F3F3Fu, (w.h[3] & 0x0F0F0F0Fu) | ((w.h[1] >> 2) & 0x30303030u)};
            const uint32_t mn[2] = {w.h[2] & 0x3F3F3F3Fu, ((w.h[3] >> 4) & 0x0F0F0F0Fu) | ((w.h[2] >> 2) & 0x30303030u)};
            float T[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const uint32_t w0 = w.q[s >> 1][0] >> (4 * (s & 1)), w1 = w.q[s >> 1][1] >> (4 * (s & 1));
                constexpr uint32_t msk = 0x000F000Fu;
                const u32x4 b = {code2(w0, msk, 0.f), code2(w0 >> 8, msk, 0.f), code2(w1, msk, 0.f), code2(w1 >> 8, msk, 0.f)};
                const float scf = (float)((sc[s >> 2] >> (8 * (s & 3))) & 0xFFu);
                const floatx4 P = prod(s, b, zero);
                if constexpr (TWO) {
                    add2(T, P, scf, scf);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) T[e] = __builtin_fmaf(scf, P[e], T[e]);
                }
            }
            // sum over the sub-blocks of m_j * sum(x): one product with the mins as f16 integers
            u32x4 bm;
#pragma unroll
            for (int i = 0; i < 4; i++)
                bm[i] = code2(__builtin_amdgcn_perm(0u, mn[i >> 1], (i & 1) ? 0x0C030C02u : 0x0C010C00u), 0xFFFFFFFFu, 0.f);
            const floatx4 U = mfma16x16x32_f16(As, bm, zero);
            const float d = f16_to_f32(w.h[0] & 0xFFFFu), dmin = f16_to_f32(w.h[0] >> 16) * 256.0f;
#pragma unroll
            for (int e = 0; e < NE; e++)
                y[e] = (d * T[e] - dmin * (TWO ? U[2 * e] + U[2 * e + 1] : U[e])) * back[e];
        } else if constexpr (FMT == NNQ_FMT_Q8_0) {
            float T[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const uint32_t w0 = w.q[s >> 1][2 * (s & 1)] ^ 0x80808080u, w1 = w.q[s >> 1][2 * (s & 1) + 1] ^ 0x80808080u;
                constexpr uint32_t msk = 0x00FF00FFu;
                const u32x4 b = {code2(w0, msk, 128.f), code2(w0 >> 8, msk, 128.f), code2(w1, msk, 128.f),
                                 code2(w1 >> 8, msk, 128.f)};
                const floatx4 P = prod(s, b, zero);
                const float d = f16_to_f32((w.h[s >> 1] >> (16 * (s & 1))) & 0xFFFFu);
                if constexpr (TWO) {
                    add2(T, P, d, d);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) T[e] = __builtin_fmaf(d, P[e], T[e]);
                }
            }
#pragma unroll
            for (int e = 0; e < NE; e++) y[e] = T[e] * back[e];
        } else {
            float T[2] = {0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; s++) {
                // pair j of v: nibbles at bits 4j and 16 + 4j of A (s even) or B, crumbs of
                // the chunk's pair 4 (s & 1) + j at bits 2 (4 (s & 1) + j) and + 16 of C
                const uint32_t N = w.q[s >> 1][s & 1], C = w.q[s >> 1][2];
                u32x4 b;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int cs = 2 * (4 * (s & 1) + j);  // crumb position
                    const uint32_t crumb = (cs <= 4 ? C << (4 - cs) : C >> (cs - 4)) & 0x00300030u;
                    b[j] = code2(((N >> (4 * j)) & 0x000F000Fu) | crumb, 0xFFFFFFFFu, 32.f);
                }
                const floatx4 P = prod(s, b, zero);
                const uint32_t sw = w.s[s >> 1] >> (16 * (s & 1));
                const float sa = (float)(int8_t)(sw & 0xFFu), sb = (float)(int8_t)((sw >> 8) & 0xFFu);
                add2(T, P, sa, sb);
            }
            const float d = f16_to_f32(w.d & 0xFFFFu);
#pragma unroll
            for (int t = 0; t < 2; t++) y[t] = (d * T[t]) * back[t];
        }
    };
    // the waves' sums of a round's tiles to y; `buf` alternates, so one barrier per round (a
    // buffer is written again only after the other one's barrier)
    auto finish = [&](int c0, int buf) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0) only: the next tile's loads stay in flight
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        const int r = tid / (NE * 64), e = (tid >> 6) % NE;
        if (r < min(RB, t_hi - c0)) {
            // tile r of the round is the work of wave group r % ng
            const float *p = red + (((size_t)buf * kFewWaves + (r % ng) * a.up) * RB * NE + (r * NE + e)) * 64 + lane;
            float y = 0.f;
            for (int w = 0; w < nu; w++) y += p[(size_t)w * RB * NE * 64];
            const int t = NE * G + e;
            const int64_t col = (int64_t)(c0 + r) * 16 + c16;
            if (t < a.m && col < a.n) {
                if (a.ks > 1) {
                    reinterpret_cast<float *>(a.y)[((int64_t)part * a.m + t) * a.n + col] = y;
                } else {
                    if (a.bias) y += a.bias[col];
                    if (a.y_bf16)
                        reinterpret_cast<uint16_t *>(a.y)[(int64_t)t * a.n + col] = (uint16_t)f32_to_bf16_bits(y);
                    else
                        reinterpret_cast<float *>(a.y)[(int64_t)t * a.n + col] = y;
                }
            }
        }
    };

    // rounds of RB tiles; in a round the wave takes tiles grp, grp + ng, ...
    int c0 = t_lo, r = grp, buf = 0;
    if (wv % a.up < nu && t_lo + grp < t_hi) {
        auto step = [&](const FewRaw<FMT> &cur, FewRaw<FMT> &nxt) {
            int nc = c0, nr = r + ng;
            if (nr >= RB) nc += RB, nr = grp;
            const bool more = nc + nr < t_hi;
            if (more) few_load<FMT>(a, nc + nr, u, lane, nxt);
            __builtin_amdgcn_sched_barrier(0);
            float y[NE];
            compute(cur, y);
            float *p = red + (((size_t)buf * kFewWaves + wv) * RB * NE + r * NE) * 64 + lane;
#pragma unroll
            for (int e = 0; e < NE; e++) p[64 * e] = y[e];
            if (nc != c0 || !more) {
                finish(c0, buf);
                c0 += RB;
                buf ^= 1;
            }
            r = nr;
            return more;
        };
        FewRaw<FMT> b0, b1;
        // x first: its wait does not include the weights', which arrive while it is converted
        XRaw x;
        x_load(u, x);
        __builtin_amdgcn_sched_barrier(0);
        few_load<FMT>(a, c0 + r, u, lane, b0);
        __builtin_amdgcn_sched_barrier(0);
        x_stage(x);
        while (step(b0, b1) && step(b1, b0)) {
        }
    }
    // rounds in which the wave has no tile: it only joins their sums
    for (; c0 < t_hi; c0 += RB, buf ^= 1) finish(c0, buf);
}

// y = the K parts' slabs summed in order, plus the bias
__global__ __launch_bounds__(256) void few_sum_kernel(const float *slabs, int ks, const float *bias, void *y, int y_bf16,
                                                      int64_t mn, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= mn) return;
    float v = slabs[i];
    for (int s = 1; s < ks; s++) v += slabs[(int64_t)s * mn + i];
    if (bias) v += bias[i % n];
    if (y_bf16)
        reinterpret_cast<uint16_t *>(y)[i] = (uint16_t)f32_to_bf16_bits(v);
    else
        reinterpret_cast<float *>(y)[i] = v;
}

template <int FMT, int XM>
int launch_few_t(const FewArgs &f, int grid, hipStream_t st) {
    constexpr int LDS = 2 * kFewWaves * kFewRB * (FMT == NNQ_FMT_Q6_K || XM == kFewPairs ? 2 : 4) * 64 * 4;
    static bool attr_set = false;  // idempotent attribute write; races only repeat it
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_few_kernel<FMT, XM>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
        attr_set = true;
    }
    hipLaunchKernelGGL((gemm_few_kernel<FMT, XM>), dim3((unsigned)grid), dim3(kFewWaves * 64), LDS, st, f);
    return (int)hipGetLastError();
}

}  // namespace

// rows of one launch: one 16-row operand, of which a Q6_K token takes two rows
int gemm_few_rows(int fmt) { return fmt == NNQ_FMT_Q6_K ? 8 : 16; }

static int few_units(const GemmArgs &a, int fmt) { return (int)(fmt == NNQ_FMT_Q8_0 ? a.nblk / 8 : a.nblk); }

size_t gemm_few_scratch_bytes(const GemmArgs &a, int fmt) {
    const int64_t ks = (few_units(a, fmt) + kFewWaves - 1) / kFewWaves;
    return ks > 1 ? (size_t)ks * a.m * a.n * 4 : 0;
}

static int launch_few(const FewArgs &f, int fmt, bool x_bf16, int grid, hipStream_t st) {
    switch (fmt) {
    case NNQ_FMT_Q4_K:
        if (x_bf16) return launch_few_t<NNQ_FMT_Q4_K, kFewBf16>(f, grid, st);
        return f.m <= 8 ? launch_few_t<NNQ_FMT_Q4_K, kFewPairs>(f, grid, st)
                        : launch_few_t<NNQ_FMT_Q4_K, kFewPlanes>(f, grid, st);
    case NNQ_FMT_Q8_0:
        if (x_bf16) return launch_few_t<NNQ_FMT_Q8_0, kFewBf16>(f, grid, st);
        return f.m <= 8 ? launch_few_t<NNQ_FMT_Q8_0, kFewPairs>(f, grid, st)
                        : launch_few_t<NNQ_FMT_Q8_0, kFewPlanes>(f, grid, st);
    case NNQ_FMT_Q6_K:
        return x_bf16 ? launch_few_t<NNQ_FMT_Q6_K, kFewBf16>(f, grid, st)
                      : launch_few_t<NNQ_FMT_Q6_K, kFewPlanes>(f, grid, st);
    }
    return (int)hipErrorInvalidValue;
}

int launch_gemm_few(const GemmArgs &a, int fmt, void *stream) {
    if (a.m <= 0 || a.m > gemm_few_rows(fmt)) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    FewArgs f;
    f.qs = a.qs;
    f.hdr = a.hdr;
    f.x = a.x;
    f.m = (int)a.m;
    f.units = few_units(a, fmt);
    f.ntile = (int)a.ntile;
    f.ks = (f.units + kFewWaves - 1) / kFewWaves;
    const int most = (f.units + f.ks - 1) / f.ks;  // units of a workgroup
    f.up = most <= 4 ? 4 : most <= 8 ? 8 : 16;
    f.k = a.k;
    f.n = a.n;
    f.y = f.ks > 1 ? a.scratch : a.y;
    f.y_bf16 = a.y_bf16;
    f.bias = a.bias;
    // one workgroup per CU (128 registers, 16 waves), fewer when there are fewer tiles
    const int runs = (int)std::min<int64_t>(a.ntile, std::max(1, 256 / f.ks));
    int e = launch_few(f, fmt, a.x_bf16 != 0, runs * f.ks, st);
    if (e || f.ks == 1) return e;
    const int64_t mn = a.m * a.n;
    hipLaunchKernelGGL(few_sum_kernel, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<const float *>(a.scratch), f.ks, a.bias, a.y, a.y_bf16, mn, a.n);
    return (int)hipGetLastError();
}

}  // namespace nnq
