// Prefill GEMM for Q6_K weights and bf16 activations on gfx950 (more than 128 rows):
// Y[m, n] = X[m, k] . W[n, k]^T (+ bias) over load-time decoded Q6_K weights
// (crates/nn-gguf/src/dequant.rs:415-459 feeding Linear, crates/nn-core/src/layers/
// core_layers.rs:118-135; the bf16 result dtype of crates/nn-core/src/dyn_tensor/ops/matmul.rs:37-38).
//
// Arithmetic: w = d * sc_j * q' with q' = q - 32 and a scale per 16 k.  sc_j * q' needs up to 13
// bits, so it enters the f16 MFMA as two exact operands, sc_j * (q' & ~1) and sc_j * (q' & 1)
// (|sc_j| * |q' >> 1| <= 2048), two MFMAs per 16 x 16 x 32 step.  The products of a super-block
// accumulate from zero and d * partial is added to f32 totals at its end.  The activation is the
// wide Q4_K kernel's staged f16 plane (x * 2^s_row, exact for bf16 x, fragment-major).
//
// MFMA-bound (4 * M * N * K operations: 103 G at 512 x 4096 x 12288, about 110 us at the rate the
// chip holds with random f16 operands), so the tile is chosen for operand reuse: 256 rows x 128
// columns per workgroup of eight waves, 4 (M) x 2 (N), a wave tile of 64 x 64.  A B fragment read
// from LDS then serves four MFMAs and an A fragment, read from L2 into registers, eight; both
// paths run at half their width.  A workgroup decodes each weight once: per half super-block
// (128 k) its 8 tiles' two operands (64 KB) into one of two LDS buffers while the MFMAs of the
// other half run, a wave taking two (tile, 64-k chunk) pieces whose raw bytes were loaded half a
// super-block earlier.  One barrier per half.  K is split over workgroups (f32 slabs summed in
// order) when the tiles alone would leave CUs idle.
// 512 x 4096 x 12288 with staging and slab sum: 134 us in the block kernel (128 x 128 tiles, every
// wave decoding its own columns), 105 here, 980 TFLOP/s of MFMA work.
#include "nnq_device.h"
#include "nnq_internal.h"

namespace nnq {

namespace {

constexpr int NTH = 512;   // eight waves
constexpr int MT = 4;      // 16-row tiles of a wave
constexpr int NT = 4;      // 16-column tiles of a wave
constexpr int BM = 256;    // 4 waves
constexpr int TL = 8;      // weight tiles per workgroup (2 waves)
constexpr int BN = TL * 16;
constexpr int HB = TL * 4 * 2 * 1024;  // a half super-block's operands: tiles x steps x 2 x 1 KB
constexpr int D_OFF = 2 * HB;          // d of each column, f32, for two super-blocks
constexpr int OUT = BM * (BN * 4 + 16);  // the output tile, rows padded by 16 bytes
constexpr int LDS6 = OUT > D_OFF + 2 * BN * 4 ? OUT : D_OFF + 2 * BN * 4;
static_assert(LDS6 <= 160 * 1024, "LDS budget of a gfx950 workgroup");

typedef _Float16 h2 __attribute__((ext_vector_type(2)));

struct Wide6Args {
    const uint8_t *qs, *hdr;
    const u32x4 *xa;       // staged activation [row group][k / 32][16 rows][4 x 16 B]
    const float *rowback;  // [row groups * 16] 2^-s_row
    const float *bias;
    void *y;
    float *ysplit;         // [ks][m][n] f32 slabs when ks > 1
    int y_bf16;
    int m, nblk, ntile, ks, nrg;
    int64_t n;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc6(const void *p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)min(bytes, (int64_t)0x7FFFFFF0), 0x00020000);
}

__global__ __launch_bounds__(NTH, 1) void gemm_q6k_wide_kernel(Wide6Args a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wv >> 1, wn = wv & 1;
    const int G = lane >> 4, c16 = lane & 15;
    const int nblk = a.nblk;

    // tile order as in the wide Q4_K kernel: each XCD gets a contiguous run, the column tiles of
    // one row tile
    const int nct = a.ntile / TL, nrt = (a.m + BM - 1) / BM, total = nct * nrt * a.ks;
    const int bid = (int)blockIdx.x;
    const int T = (total % 8 == 0) ? (bid % 8) * (total / 8) + bid / 8 : bid;
    const int kp = T / (nct * nrt), Tt = T % (nct * nrt);
    const int rt = Tt / nct, ct = Tt % nct;
    const int t0 = ct * TL, nsb = nblk / a.ks, sb0 = kp * nsb;

    // A fragments: the wave's four row groups (past the last: clamped, not stored)
    __amdgpu_buffer_rsrc_t ra[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int rg = min(rt * (BM / 16) + wm * MT + mt, a.nrg - 1);
        ra[mt] = rsrc6(a.xa + ((size_t)rg * nblk * 8 + (size_t)sb0 * 8) * 64, (int64_t)nsb * 8 * 1024);
    }
    const int loff = (c16 * 4 + G) * 16;
    // decode pieces of a half: wave w takes tile w, chunks 2h and 2h + 1 (64 k each)
    const __amdgpu_buffer_rsrc_t rq = rsrc6(a.qs + ((size_t)(t0 + wv) * nblk + sb0) * 3072, (int64_t)nsb * 3072);
    const __amdgpu_buffer_rsrc_t rh = rsrc6(a.hdr + ((size_t)(t0 + wv) * nblk + sb0) * 288, (int64_t)nsb * 288);
    u32x3 raw[2];
    uint32_t rsc[2], rd;
    const int nh = 2 * nsb;  // halves
    auto load_raw = [&](int h) {
        const int sb = h >> 1, c0 = 2 * (h & 1);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            raw[j] = __builtin_bit_cast(
                u32x3, __builtin_amdgcn_raw_buffer_load_b96(rq, 12 * lane, sb * 3072 + (c0 + j) * 768, 0));
            rsc[j] = __builtin_amdgcn_raw_buffer_load_b32(rh, 16 * c16, sb * 288 + 4 * (c0 + j), 0);
        }
        rd = __builtin_amdgcn_raw_buffer_load_b16(rh, 256 + 2 * c16, sb * 288, 0);
    };
    // piece j of half h: lane (G, row c16) decodes its 8 codes of steps 2j and 2j + 1 into the two
    // operands.  Pair i of a step: nibbles at bits 4i and 16 + 4i of word A or B, crumbs at bits
    // 2 (4 e + i) and + 16 of word C (e: the step's parity)
    auto store_piece = [&](int h, int j) {
        unsigned char *buf = smem + (h & 1) * HB + (wv * 4 + 2 * j) * 2048 + lane * 16;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            // the lane group's scale: sub-block 2 e + (G >> 1) of the chunk, as f16 in both halves
            // (0x6480 ^ byte is 1152 + s exactly)
            const uint32_t sb8 = (rsc[j] >> (16 * e + 8 * (G >> 1))) & 0xFFu;
            const h2 sc = __builtin_bit_cast(h2, (sb8 | (sb8 << 16)) ^ 0x64806480u) +
                          h2{(_Float16)-1152.0f, (_Float16)-1152.0f};
            const uint32_t N = raw[j][e], C = raw[j][2];
            u32x4 b0, b1;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int cs = 2 * (4 * e + i);
                const uint32_t q = ((N >> (4 * i)) & 0x000F000Fu) |
                                   ((cs <= 4 ? C << (4 - cs) : C >> (cs - 4)) & 0x00300030u);
                const h2 ev = __builtin_bit_cast(h2, (q & 0x003E003Eu) | 0x64006400u) +
                              h2{(_Float16)-1056.0f, (_Float16)-1056.0f};  // (q' & ~1)
                const h2 od = __builtin_bit_cast(h2, (q & 0x00010001u) | 0x64006400u) +
                              h2{(_Float16)-1024.0f, (_Float16)-1024.0f};  // q' & 1
                b0[i] = __builtin_bit_cast(uint32_t, ev * sc);
                b1[i] = __builtin_bit_cast(uint32_t, od * sc);
            }
            *reinterpret_cast<u32x4 *>(buf + e * 2048) = b0;
            *reinterpret_cast<u32x4 *>(buf + e * 2048 + 1024) = b1;
        }
        if (j == 0 && !(h & 1) && G == 0)
            *reinterpret_cast<float *>(smem + D_OFF + ((h >> 1) & 1) * BN * 4 + (wv * 16 + c16) * 4) = f16_to_f32(rd & 0xFFFFu);
    };

    floatx4 tot[MT][NT], part[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) tot[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};

    load_raw(0);
    u32x4 af[2][MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
        af[0][mt] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ra[mt], loff, 0, 0));
    store_piece(0, 0);
    store_piece(0, 1);
    load_raw(1);  // (every super-block has two halves)
    auto sync = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's LDS reads and writes
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    sync();

    for (int sb = 0; sb < nsb; sb++) {
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
            const int h = 2 * sb + hf;
            const unsigned char *cur = smem + hf * HB + wn * NT * 8192;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int gs = h * 4 + s;
                // the next step's A fragments (past the range: zeros, never used)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    af[(s + 1) & 1][mt] = __builtin_bit_cast(
                        u32x4, __builtin_amdgcn_raw_buffer_load_b128(ra[mt], loff, (gs + 1) * 1024, 0));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n0 = 0; n0 < NT; n0 += 2) {
                    u32x4 bf[2][2];
#pragma unroll
                    for (int j = 0; j < 2; j++)
#pragma unroll
                        for (int o = 0; o < 2; o++)
                            bf[j][o] = *reinterpret_cast<const u32x4 *>(cur + ((n0 + j) * 4 + s) * 2048 + o * 1024 + lane * 16);
#pragma unroll
                    for (int o = 0; o < 2; o++)
#pragma unroll
                        for (int j = 0; j < 2; j++)
#pragma unroll
                            for (int mt = 0; mt < MT; mt++)
                                part[mt][n0 + j] = mfma16x16x32_f16(af[s & 1][mt], bf[j][o],
                                                                    hf == 0 && s == 0 && o == 0
                                                                        ? floatx4{0.f, 0.f, 0.f, 0.f}
                                                                        : part[mt][n0 + j]);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // the next half's operands into the other buffer (read by nobody since the barrier
                // that ended the previous half), then its successor's raw bytes
                if (s >= 1 && s < 3 && h + 1 < nh) store_piece(h + 1, s - 1);
                if (s == 2 && h + 2 < nh) load_raw(h + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (hf == 1) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const float dn = *reinterpret_cast<const float *>(smem + D_OFF + (sb & 1) * BN * 4 +
                                                                      ((wn * NT + nt) * 16 + c16) * 4);
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
#pragma unroll
                        for (int e = 0; e < 4; e++) tot[mt][nt][e] += dn * part[mt][nt][e];
                }
            }
            sync();
        }
    }

    // epilogue: y = tot * 2^-s_row (+ bias), assembled in LDS and written as 16-byte row chunks
    const bool f32out = a.ks > 1 || !a.y_bf16;
    const int es = f32out ? 4 : 2, rs = BN * es + 16;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const floatx4 rb = *reinterpret_cast<const floatx4 *>(
            a.rowback + min(rt * BM + wm * 64 + mt * 16, a.nrg * 16 - 16) + 4 * G);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int col = (wn * NT + nt) * 16 + c16;
            const float bc = (a.bias && a.ks == 1) ? a.bias[(int64_t)t0 * 16 + col] : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float y = tot[mt][nt][e] * rb[e] + bc;
                unsigned char *p = smem + (wm * 64 + mt * 16 + 4 * G + e) * rs + col * es;
                if (f32out)
                    *reinterpret_cast<float *>(p) = y;
                else
                    *reinterpret_cast<uint16_t *>(p) = (uint16_t)f32_to_bf16_bits(y);
            }
        }
    }
    __syncthreads();
    const int cpr = BN * es / 16, m0 = rt * BM;
    unsigned char *ybase = a.ks > 1 ? reinterpret_cast<unsigned char *>(a.ysplit + (int64_t)kp * a.m * a.n)
                                    : reinterpret_cast<unsigned char *>(a.y);
    for (int c = tid; c < BM * cpr; c += NTH) {
        const int rl = c / cpr, ch = c - rl * cpr;
        if (m0 + rl >= a.m) break;  // rows run in order
        *reinterpret_cast<u32x4 *>(ybase + ((int64_t)(m0 + rl) * a.n + (int64_t)t0 * 16) * es + ch * 16) =
            *reinterpret_cast<const u32x4 *>(smem + rl * rs + ch * 16);
    }
}

}  // namespace

// The K split (0: the block kernel takes the call): the rule of its shape (nnq_rule_gemm_wide6), for
// Q6_K, bf16 activations, whole 16-row weight tiles and a 16-byte aligned output.
int gemm_wide6_plan(const GemmArgs &a) {
    if (a.blk != NNQ_FMT_Q6_K || !a.x_bf16 || a.n != a.ntile * 16 || (reinterpret_cast<uintptr_t>(a.y) & 15)) return 0;
    return nnq_rule_gemm_wide6(a.m, a.ntile, a.nblk);
}

// scratch: the staged activation | rowback | slabs
size_t gemm_wide6_scratch(const GemmArgs &a, GemmScratch *s, uint8_t *base) {
    auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
    const int64_t nrg = (a.m + 15) / 16;
    const int ks = gemm_wide6_plan(a);
    const size_t xb = al((size_t)nrg * 16 * a.k * 2), rb = al((size_t)nrg * 16 * 4);
    if (s) {
        s->xh = reinterpret_cast<uint16_t *>(base);
        s->xs = nullptr;
        s->rowback = reinterpret_cast<float *>(base + xb);
        s->ksplit = ks;
        s->ysplit = ks > 1 ? reinterpret_cast<float *>(base + xb + rb) : nullptr;
    }
    return xb + rb + (ks > 1 ? al((size_t)ks * a.m * a.n * 4) : 0);
}

int launch_gemm_wide6(const GemmArgs &a, const GemmScratch &sc, void *stream) {
    const int ks = gemm_wide6_plan(a);
    if (!ks || sc.ksplit != ks || (ks > 1 && !sc.ysplit)) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    int e = launch_stage_wide(a.x, 1, a.m, a.k, sc.xh, nullptr, sc.rowback, stream);
    if (e) return e;
    static bool attr_set = false;  // idempotent attribute write; races only repeat it
    if (!attr_set) {
        hipError_t he = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_q6k_wide_kernel),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, LDS6);
        if (he != hipSuccess) return (int)he;
        attr_set = true;
    }
    Wide6Args w{};
    w.qs = a.qs;
    w.hdr = a.hdr;
    w.xa = reinterpret_cast<const u32x4 *>(sc.xh);
    w.rowback = sc.rowback;
    w.bias = a.bias;
    w.y = a.y;
    w.ysplit = sc.ysplit;
    w.y_bf16 = a.y_bf16;
    w.m = (int)a.m;
    w.n = a.n;
    w.nblk = (int)a.nblk;
    w.ntile = (int)a.ntile;
    w.ks = ks;
    w.nrg = (int)((a.m + 15) / 16);
    const int total = (w.ntile / TL) * ((w.m + BM - 1) / BM) * ks;
    hipLaunchKernelGGL(gemm_q6k_wide_kernel, dim3((unsigned)total), dim3(NTH), LDS6, st, w);
    e = (int)hipGetLastError();
    if (e || ks == 1) return e;
    return launch_gemm_finalize(sc.ysplit, ks, a.bias, a.y, a.y_bf16, a.m, a.n, stream);
}

}  // namespace nnq
