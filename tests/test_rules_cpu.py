"""The rules that choose a kernel by sizes alone (nn_amd/csrc/nnq_plan.cpp), asked through their C names:
what holds for every shape.  No GPU needed."""
import random

import pytest

Q8_0, Q4_K, Q6_K = 8, 12, 14

def test_kernel_limits(rules):
    """No rule sends a kernel what it cannot run: rows of the few-row GEMM, tiles and K parts that divide
    the weight, two super-blocks a part, the staging's K, the few-token kernel's ballots and rows."""
    rng = random.Random(3)
    for _ in range(20000):
        m, tiles, nblk, bf16 = rng.randint(1, 3000), rng.randint(1, 4096), rng.randint(1, 64), rng.randint(0, 1)
        n, k = 16 * tiles, 256 * nblk
        nt, ks = rules.wide(m, n, k, bf16)
        if nt:
            assert m > 128 and k <= 12288 and nt in (4, 6, 8) and tiles % nt == 0 and nblk % ks == 0 and nblk // ks >= 2
        ks = rules.wide6(m, n, k)
        if ks:
            assert m > 128 and k <= 12288 and tiles % 8 == 0 and nblk % ks == 0 and nblk // ks >= 2
        for fmt in (Q8_0, Q4_K, Q6_K):
            if rules.few_rows(fmt, m, n, k, bf16):
                assert 3 <= m <= 16
        experts, top_k, tokens = rng.randint(1, 300), rng.randint(1, 16), rng.randint(1, 40)
        if top_k <= experts and rules.moe_few(experts, 32 * rng.randint(1, 200), 32 * rng.randint(1, 200), tokens, top_k, bf16):
            assert tokens <= 16 and tokens * top_k <= 128


# Layers measured on both kernels, those of 1.1x or more between them (us, moe_stream_kernel / moe_few_kernel).
@pytest.mark.parametrize("experts,hidden,inter,tokens,top_k,bf16,few", [
    (32, 2880, 2880, 1, 4, 1, 1),    # 93 / 27
    (32, 2880, 2880, 8, 4, 1, 1),    # 99 / 81
    (32, 2880, 2880, 12, 8, 1, 0),   # 108 / 123
    (32, 2880, 2880, 16, 8, 1, 0),   # 109 / 151
    (32, 2880, 2880, 16, 4, 0, 0),   # 127 / 161
    (32, 2880, 2880, 16, 8, 0, 0),   # 132 / 238
    (16, 2880, 2880, 16, 4, 1, 1),   # 98 / 80
    (16, 2880, 2880, 16, 8, 1, 0),   # 101 / 126
    (16, 2880, 2880, 16, 8, 0, 0),   # 126 / 201
    (8, 2880, 2880, 12, 8, 1, 1),    # 103 / 81
    (8, 2880, 2880, 16, 8, 0, 0),    # 125 / 164
    (32, 2048, 2048, 8, 4, 1, 1),    # 92 / 61
    (32, 2048, 2048, 16, 8, 0, 0),   # 99 / 150
    (32, 768, 2880, 16, 8, 0, 0),    # 67 / 91
    (48, 2048, 1408, 16, 6, 0, 1),   # 156 / 110
    (64, 2880, 1440, 16, 8, 0, 1),   # 185 / 161
    (8, 4096, 14336, 16, 2, 0, 1),   # 985 / 352
])
def test_moe_few_where_it_is_faster(rules, experts, hidden, inter, tokens, top_k, bf16, few):
    assert rules.moe_few(experts, hidden, inter, tokens, top_k, bf16) == few


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("experts,hidden,inter,top_k", [(1, 32, 32, 1), (8, 2880, 2880, 8), (32, 2880, 2880, 4),
                                                        (4096, 32768, 32768, 8)])
def test_moe_few_is_a_limit_in_tokens(rules, experts, hidden, inter, top_k, bf16):
    """More tokens never bring the few-token kernel back, and one token always takes it."""
    got = [rules.moe_few(experts, hidden, inter, t, top_k, bf16) for t in range(1, 20)]
    assert got[0] == 1 and got == sorted(got, reverse=True) and not any(got[16:])


# Linears measured both ways, most with 1.1x or more between them (us, GEMV passes or MFMA GEMM / few-row GEMM).
@pytest.mark.parametrize("fmt,m,n,k,bf16,few", [
    (Q4_K, 3, 151936, 1024, 0, 1),   # 28.4 / 25.4
    (Q4_K, 4, 32768, 3072, 0, 1),    # 18.9 / 17.0
    (Q4_K, 3, 40960, 256, 1, 1),     # 13.3 / 10.1 (thin GEMM)
    (Q6_K, 3, 65536, 2048, 1, 1),    # 29.6 / 23.8
    (Q8_0, 3, 151936, 1024, 0, 1),   # 34.7 / 29.7
    (Q6_K, 16, 65536, 256, 0, 0),    # 18.7 / 27.1
    (Q6_K, 16, 32768, 512, 1, 0),    # 13.8 / 18.4
    (Q6_K, 16, 65536, 1024, 0, 1),   # 46.2 / 33.2
    (Q6_K, 16, 8192, 512, 1, 1),     # 13.7 / 11.3
    (Q6_K, 8, 65536, 256, 1, 1),
    (Q8_0, 16, 65536, 256, 1, 1),
    (Q4_K, 6, 4096, 4096, 0, 0),
    (Q4_K, 6, 4096, 12288, 0, 1),    # 19.0 / 17.2
    (Q4_K, 16, 12288, 4096, 1, 0),   # 10.0 / 13.0 (thin GEMM)
])
def test_few_rows_where_they_are_faster(rules, fmt, m, n, k, bf16, few):
    assert rules.few_rows(fmt, m, n, k, bf16) == few


# Q6_K prefill measured on the block and the wide kernel (us, block / wide).
@pytest.mark.parametrize("m,n,k,wide", [
    (129, 40960, 1024, 0),   # 59.4 / 66.1
    (160, 40960, 1024, 0),   # 62.1 / 66.9
    (129, 9728, 2560, 0),    # 45.7 / 47.9
    (200, 40960, 1024, 1),   # 74.6 / 67.6
    (160, 12288, 4096, 2),   # 87.0 / 68.7
    (129, 4096, 4096, 8),    # 35.3 / 31.5
    (160, 6144, 2048, 4),    # 34.8 / 31.1
    (129, 4096, 12288, 8),   # 74.3 / 56.2
    (129, 24576, 1536, 1),   # 54.9 / 49.2
    (512, 4096, 12288, 4),   # 133.8 / 103.6
])
def test_wide6_where_it_is_faster(rules, m, n, k, wide):
    assert rules.wide6(m, n, k) == wide


# Q4_K prefill measured with other tiles and splits (us, what the rule takes / the other one named).
@pytest.mark.parametrize("m,n,k,bf16,tiles,split", [
    (400, 2560, 2560, 1, 4, 2),    # 25.0 / 27.9 with 8 tiles, K in five
    (512, 2560, 2560, 1, 4, 2),    # 27.2 / 29.5 with 8 tiles, K in five
    (200, 6144, 2048, 1, 4, 2),    # 23.6 / 25.4 with 6 tiles, K in four
    (129, 8192, 3072, 1, 4, 2),    # 26.6 / 28.7 with 8 tiles, K in four
    (768, 4096, 12288, 1, 8, 2),   # 109.6 / 118.6 with 8 tiles, K in eight
    (512, 4096, 12288, 1, 8, 4),   # 69.0 / 77 with 4 tiles, K in two
    (512, 4096, 12288, 0, 8, 4),   # 105.1 / 142.1 in the ring kernel
    (203, 12288, 4096, 0, 6, 2),   # 57.9 / 74.0 in the ring kernel
    (512, 24576, 4096, 1, 6, 1),
    (260, 5376, 11008, 0, 0, 0),   # ring kernel 124.6 / 186.9 with 4 tiles (43 super-blocks cannot be split)
    (384, 5376, 11008, 0, 0, 0),   # ring kernel 127.0 / 188.0
    (600, 5376, 11008, 0, 4, 1),   # 194.8 / 231.4 in the ring kernel
    (384, 4736, 1792, 0, 0, 0),    # ring kernel 34.1 / 39.2 with 4 tiles
    (600, 4736, 1792, 0, 4, 1),    # 40.8 / 54.8 in the ring kernel
    (260, 5376, 11008, 1, 4, 1),   # 108.5 / 119.5 in the ring kernel
])
def test_wide_tiles_where_they_are_faster(rules, m, n, k, bf16, tiles, split):
    assert rules.wide(m, n, k, bf16) == (tiles, split)


# f32 prefill MLPs measured with either kernel under their gate | up (us, ring kernel and SwiGLU launch / wide kernel).
@pytest.mark.parametrize("m,hidden,inter,wide", [
    (260, 768, 2048, 4),    # 49.5 / 44.3
    (260, 1024, 2560, 4),   # 49.9 / 47.7
    (129, 1792, 4608, 4),   # 66.3 / 61.4
    (260, 3328, 4864, 8),   # 151.8 / 146.5
    (260, 1792, 2560, 0),   # 62.4 / 66.1
    (129, 2816, 4096, 0),   # 71.5 / 78.3
    (260, 3328, 8704, 0),   # 251.0 / 258.5
])
def test_wide_swiglu_where_it_is_faster(rules, m, hidden, inter, wide):
    """The launch that the ring kernel's MLP has more is counted, in calls that can write h themselves only."""
    assert rules.wide(m, 2 * inter, hidden, 0, 1)[0] == wide
    assert rules.wide(m, 2 * inter, hidden, 0) == (0, 0)
