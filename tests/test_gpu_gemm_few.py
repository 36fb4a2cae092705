"""GPU parity of the few-row GEMM (3 .. 16 token rows over one read of the weight) against the
device's own bit-exact decode (tests/test_gpu_linear.py) and a float64 product, at the edges of
its rules: 5, 8, 9 and 16 rows (one and two launches of Q6_K, f32 operands as row pairs or as
planes), 3 rows over 2048 tiles; N below a tile, past one, and an uneven number of tiles per
workgroup; K of 1, 4, 8, 9, 16, 17 and 33 units of 256 (one to four wave groups, K split two and
three ways) and, for Q8_0, K that ends inside a unit.  Q4_K with bf16 x takes this kernel from 2048
tiles on, so its shapes have a row count of their own.

Bar: products are exact in f32 (f32 x: its hi + lo f16 pair drops 2^-22 of it), so what is left is
the rounding of f32 sums, 2^-24 of partial sums that stay within a few times the output's own
size: max |error| <= 1e-5 of the output's root mean square (some 40 roundings in line)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(8, 7, 256), (5, 300, 1024), (16, 40, 2048), (9, 1000, 2304), (8, 4112, 4096), (16, 65, 4352), (7, 33, 8448),
          (3, 32784, 512), (12, 2080, 768)]


def weight(fmt, n, k, seed):
    import nn_amd
    w = nn_amd.synth_normal(seed, 1, (n, k), 0.02)
    quant = {"q8_0": nn_amd.quantize_q8_0, "q4_k": nn_amd.quantize_q4_k, "q6_k": nn_amd.quantize_q6_k}[fmt]
    qt = {"q8_0": nn_amd.QuantType.Q8_0, "q4_k": nn_amd.QuantType.Q4_K, "q6_k": nn_amd.QuantType.Q6_K}[fmt]
    layout = nn_amd.Layout.NN_GGUF if fmt == "q6_k" else nn_amd.Layout.GGUF
    return nn_amd.QuantizedWeight.from_quantized(quant(w), qt, (n, k), layout=layout)


def check(y, ref, what):
    err = (y.double() - ref).abs().max().item() / ref.pow(2).mean().sqrt().item()
    assert err <= 1e-5, f"{what}: max error {err:.2e} of the output's rms"


QT = {"q8_0": 8, "q4_k": 12, "q6_k": 14}
CELLS = [(m, n, k, fmt, xdt) for m, n, k in SHAPES for fmt in QT for xdt in (torch.float32, torch.bfloat16)
         if n >= 32768 or not (fmt == "q4_k" and xdt == torch.bfloat16)]
# rows 4 .. 16, one, two and four wave groups, several units a group, K split evenly and unevenly,
# a last tile of one row
CELLS += [(m, n, k, "q4_k", torch.bfloat16) for m, n, k in
          ((4, 32753, 256), (5, 33000, 1024), (9, 32784, 2304), (16, 32784, 4096), (13, 33000, 4352), (7, 32768, 8448))]


def tall_weight(fmt, n, k, seed):
    """A weight of many rows: 1007 quantized ones over and over (no whole number of tiles)."""
    import nn_amd
    if n <= 4200:
        return weight(fmt, n, k, seed)
    quant = {"q8_0": nn_amd.quantize_q8_0, "q4_k": nn_amd.quantize_q4_k, "q6_k": nn_amd.quantize_q6_k}[fmt]
    rows = np.asarray(quant(nn_amd.synth_normal(seed, 1, (1007, k), 0.02))).reshape(1007, -1)
    layout = nn_amd.Layout.NN_GGUF if fmt == "q6_k" else nn_amd.Layout.GGUF
    b = np.ascontiguousarray(rows[np.arange(n) % 1007]).ravel()
    return nn_amd.QuantizedWeight.from_quantized(b, nn_amd.QuantType(QT[fmt]), (n, k), layout=layout)


@pytest.mark.parametrize("m,n,k,fmt,xdt", CELLS)
def test_few_rows(rules, m, n, k, fmt, xdt):
    import nn_amd
    nn_amd.init(0)
    if m > 6 or n >= 32768 or fmt != "q4_k":  # (Q4_K with f32 x: from 7 rows at these sizes)
        assert rules.few_rows(QT[fmt], m, n, k, xdt == torch.bfloat16) == 1
    qw = tall_weight(fmt, n, k, 31 + n)
    x = torch.from_numpy(nn_amd.synth_normal(33, m, (m, k), 1.0)).cuda().to(xdt)
    bias = torch.from_numpy(nn_amd.synth_normal(33, 3, (n,), 0.1)).cuda()
    ref = x.double() @ qw.dequantize().double().t() + bias.double()
    y = nn_amd.quantized_linear(x, qw, bias)
    check(y, ref, f"{fmt} {m}x{n}x{k} {xdt}")
    yb = nn_amd.quantized_linear(x, qw, bias, out_dtype=torch.bfloat16)
    assert torch.equal(yb, y.to(torch.bfloat16)), "bf16 output is the f32 result rounded once"


# More than 8 rows of Q6_K are two launches: four tiles per CU of one or two units take the MFMA GEMM
# instead (one tile below the limit, at it, and past it with a ragged last tile).
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(9, 16368, 512), (9, 16369, 512), (16, 16400, 256), (12, 16384, 768)])
def test_q6_k_two_launches_or_gemm(m, n, k, xdt):
    import nn_amd
    nn_amd.init(0)
    qw = weight("q6_k", n, k, 45)
    x = torch.from_numpy(nn_amd.synth_normal(47, m, (m, k), 1.0)).cuda().to(xdt)
    check(nn_amd.quantized_linear(x, qw), x.double() @ qw.dequantize().double().t(), f"q6_k {m}x{n}x{k} {xdt}")


@pytest.mark.parametrize("m,n,k", [(5, 300, 96), (16, 40, 4128), (8, 64, 4096 + 32), (13, 48, 8192 + 224)])
def test_few_rows_q8_0_partial_unit(m, n, k):
    import nn_amd
    nn_amd.init(0)
    qw = weight("q8_0", n, k, 35)
    big = torch.from_numpy(nn_amd.synth_normal(37, m, (m, k), 1.0)).cuda()
    for x in (big, big.to(torch.bfloat16)):
        check(nn_amd.quantized_linear(x, qw), x.double() @ qw.dequantize().double().t(), f"q8_0 {m}x{n}x{k}")


@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("fmt", ["q8_0", "q4_k", "q6_k"])
def test_few_rows_magnitudes_and_nonfinite_rows(rules, fmt, xdt):
    """Rows scaled from 1e-30 to 1e30 keep their relative accuracy; a NaN or an infinity turns its own
    row, and no other, into NaN."""
    import nn_amd
    nn_amd.init(0)
    n, k = 32784 if fmt == "q4_k" and xdt == torch.bfloat16 else 96, 1280
    assert rules.few_rows(QT[fmt], 8, n, k, xdt == torch.bfloat16) == 1
    qw = tall_weight(fmt, n, k, 39)
    x = torch.from_numpy(nn_amd.synth_normal(41, 1, (8, k), 1.0)).cuda()
    x *= torch.tensor([1e-30, 1e30, 1.0, 0.0, 1e-10, 1e10, 1.0, 1.0], device=x.device)[:, None]
    x[2, ::2] *= 1e-6  # a wide range inside each unit
    x = x.to(xdt)
    ref = x.double() @ qw.dequantize().double().t()
    y = nn_amd.quantized_linear(x, qw)
    for i in range(8):
        if i != 3:
            check(y[i], ref[i], f"{fmt} row {i}")
    assert not y[3].any()
    x[6, 100], x[7, 1279] = float("nan"), float("-inf")
    z = nn_amd.quantized_linear(x, qw)
    assert torch.equal(z[:6], y[:6])
    assert torch.isnan(z[6:]).all()
