"""GPU parity for the Q4_K prefill GEMMs of bf16 activations at every batch size the
random-byte shapes below reach: the wide-wave-tile kernel (more than 128 rows), the
skinny kernel (17 to 32 rows over three tiles per workgroup), the one-launch thin kernel
(up to 16 rows) and the ring kernel between them, against the oracle's bit-exact decode
followed by an f64 product (tolerances as in test_gpu_linear).  Shapes cover both wide
column-tile widths (96 columns, and 64 with the K range split in two), ragged row tiles
(the last tile partly past M, a row group partly past M), random block bytes (arbitrary
finite d / dmin / scales, with d = 0 super-blocks), bias, f32 and bf16 outputs, and
repeated calls agreeing bit for bit."""
import numpy as np
import pytest
import torch

from test_gpu_gemm import ref_f64
from test_gpu_linear import check_close, make_weight, rand_bytes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def dev():
    import nn_amd
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nn_amd.init(0)
    return torch.device("cuda:0")


@pytest.mark.parametrize("m,n,k", [(300, 12288, 1024), (512, 12288, 512), (129, 4096, 2048), (700, 4096, 1536),
                                   (257, 6144, 1024), (1000, 8192, 512), (5, 12288, 1024), (32, 12288, 512),
                                   (48, 12288, 1024), (64, 4096, 8192), (17, 3072, 12288), (63, 768, 2048), (40, 1528, 1024), (300, 1528, 512)])
@pytest.mark.parametrize("legacy", [False, True])
def test_wide_random_blocks(O, dev, m, n, k, legacy):
    import nn_amd
    b = rand_bytes("q4_k", n, k, seed=m * 7 + n + k).reshape(-1, 144).copy()
    b[::7, 0:2] = 0  # d = +0.0 for every seventh super-block
    b = b.ravel()
    w = make_weight("q4_k_legacy" if legacy else "q4_k", b, n, k)
    x = torch.from_numpy(nn_amd.synth_normal(m + 1, 2, (m, k), 1.0)).to(dev).to(torch.bfloat16)
    bias = torch.from_numpy(nn_amd.synth_normal(m + 1, 3, (n,), 0.5)).to(dev)
    y = nn_amd.quantized_linear(x, w, bias)
    y2 = nn_amd.quantized_linear(x, w, bias)
    assert torch.equal(y, y2), "repeated calls must agree bit for bit"
    ref = ref_f64(O, b, n, k, x.float().cpu().numpy(), legacy=legacy) + bias.cpu().numpy()
    check_close(ref, y.cpu().numpy(), f"gemm wide {m}x{n}x{k} legacy={legacy}")
    yb = nn_amd.quantized_linear(x, w, bias, out_dtype=torch.bfloat16).float().cpu().numpy()
    assert np.array_equal(yb, y.to(torch.bfloat16).float().cpu().numpy()), "bf16 output: the f32 result rounded once"


def test_wide_row_scales(O, dev):
    """Rows of very different magnitudes (1e-6 to 1e4) and a zero row: each row has its own
    power-of-two staging scale, so every row keeps its relative accuracy."""
    import nn_amd
    m, n, k = 260, 12288, 512
    wb = nn_amd.quantize_q4_k(nn_amd.synth_normal(9, 1, (n, k), 0.02))
    w = make_weight("q4_k", wb, n, k)
    xs = nn_amd.synth_normal(9, 2, (m, k), 1.0)
    xs *= (10.0 ** np.linspace(-6, 4, m)).astype(np.float32)[:, None]
    xs[17] = 0.0
    x = torch.from_numpy(xs).to(dev).to(torch.bfloat16)
    y = nn_amd.quantized_linear(x, w).cpu().numpy()
    ref = ref_f64(O, wb, n, k, x.float().cpu().numpy())
    assert np.all(y[17] == 0.0)
    keep = np.arange(m) != 17
    r, g = ref[keep], y[keep]
    # per row, normwise against that row's peak (the rows' scales differ by 10 decades)
    err = np.abs(g - r).max(axis=1) / np.abs(r).max(axis=1)
    print(f"row-scale sweep: worst per-row normwise {err.max():.2e}")
    assert err.max() <= 1e-3


def check_activations(dev, m, n, k, xdt):
    """Bar: max |error| <= 2e-5 of a row's rms: f32 sums over K <= 12288 of products that keep 22 bits of x
    (2.3e-6 measured at 512 x 4096 x 12288)."""
    import nn_amd
    w = make_weight("q4_k", nn_amd.quantize_q4_k(nn_amd.synth_normal(m, 1, (n, k), 0.02)), n, k)
    x = torch.from_numpy(nn_amd.synth_normal(m, 2, (m, k), 1.0)).to(dev)
    x[5] *= 1e-20
    x[7] = 0.0
    x = x.to(xdt)
    bias = torch.from_numpy(nn_amd.synth_normal(m, 3, (n,), 0.5)).to(dev)
    y = nn_amd.quantized_linear(x, w, bias)
    assert torch.equal(y, nn_amd.quantized_linear(x, w, bias)), "repeated calls must agree bit for bit"
    ref = x.double() @ w.dequantize().double().t() + bias.double()
    err = ((y.double() - ref).abs().amax(1) / ref.pow(2).mean(1).sqrt()).max().item()
    assert err <= 2e-5, f"{m}x{n}x{k}: {err:.2e} of the row's rms"
    yb = nn_amd.quantized_linear(x, w, bias, out_dtype=torch.bfloat16)
    assert torch.equal(yb, y.to(torch.bfloat16)), "bf16 output: the f32 result rounded once"


# f32 and bf16 activations from the wide kernel's lower limit on, ragged row tiles, K up to the
# staging's limit.  (129 x 3072 x 1024 and 700 x 1920 x 768 are too few workgroups for the wide kernel:
# the ring kernel at the same row counts.)
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(129, 3072, 1024), (203, 12288, 512), (300, 6144, 2048), (513, 4096, 1280),
                                   (256, 2048, 12288), (700, 1920, 768), (512, 4096, 2048), (1100, 4096, 512),
                                   (1000, 2048, 2560)])
def test_wide_activations(dev, m, n, k, xdt):
    check_activations(dev, m, n, k, xdt)


# Every instantiation of the wide kernel, with and without a K split: one row past the lower limit, a row
# past one and two row tiles; parts of two super-blocks (the fewest), and of three and more, where the
# ring of min-term operands wraps.  The rule has to give the tiles and the split named here.
@pytest.mark.parametrize("xdt,m,n,k,tiles,split", [
    ("f32", 129, 1024, 4096, 4, 8), ("f32", 257, 4096, 512, 4, 1), ("f32", 513, 6144, 512, 6, 1),
    ("f32", 257, 3072, 1536, 6, 3), ("f32", 203, 6144, 4096, 6, 4), ("f32", 513, 8192, 512, 8, 1),
    ("f32", 513, 4096, 2048, 8, 2), ("f32", 257, 2048, 2560, 8, 5), ("bf16", 129, 1024, 4096, 4, 8),
    ("bf16", 257, 4096, 1280, 4, 1), ("bf16", 257, 2048, 2048, 4, 4), ("bf16", 513, 6144, 512, 6, 1),
    ("bf16", 257, 3072, 3072, 6, 4), ("bf16", 513, 8192, 512, 8, 1), ("bf16", 513, 3072, 3072, 8, 3),
    ("bf16", 513, 2048, 4096, 8, 4)])
def test_wide_tiles_and_splits(dev, rules, xdt, m, n, k, tiles, split):
    assert rules.wide(m, n, k, xdt == "bf16") == (tiles, split)
    check_activations(dev, m, n, k, torch.bfloat16 if xdt == "bf16" else torch.float32)


@pytest.mark.parametrize("m,n,k,tiles", [(129, 1024, 4096, 4), (203, 6144, 4096, 6), (513, 4096, 2048, 8)])
def test_wide_f32_random_blocks(O, dev, rules, m, n, k, tiles):
    """Random block bytes (any finite d, dmin and scales) with f32 x, whose codes the kernel forms as
    normal f16 numbers; bars of test_gpu_linear."""
    import nn_amd
    assert rules.wide(m, n, k, 0)[0] == tiles
    b = rand_bytes("q4_k", n, k, seed=m + n + k).reshape(-1, 144).copy()
    b[::7, 0:2] = 0  # d = +0.0 for every seventh super-block
    b = b.ravel()
    w = make_weight("q4_k", b, n, k)
    x = nn_amd.synth_normal(m + 1, 2, (m, k), 1.0)
    y = nn_amd.quantized_linear(torch.from_numpy(x).to(dev), w).cpu().numpy()
    check_close(ref_f64(O, b, n, k, x), y, f"gemm wide f32 {m}x{n}x{k}")


@pytest.mark.parametrize("m,hidden,inter,xdt", [(129, 512, 6144, torch.bfloat16), (300, 1024, 3072, torch.float32),
                                               (260, 768, 2048, torch.float32), (600, 512, 2048, torch.bfloat16)])
def test_prefill_mlp_swiglu_epilogue(dev, rules, m, hidden, inter, xdt):
    """The gate | up GEMM that writes silu(gate) * up itself, against the three linears: h differs by
    f32 rounding only, so the outputs agree to 1e-5 of their rms; a NaN row is flagged and stays
    in its row."""
    import nn_amd
    assert rules.wide(m, 2 * inter, hidden, xdt == torch.bfloat16, 1)[1] == 1  # the wide kernel, K not split
    q = [nn_amd.quantize_q4_k(nn_amd.synth_normal(5, i, s, 0.02))
         for i, s in ((1, (inter, hidden)), (2, (inter, hidden)), (3, (hidden, inter)))]
    mlp = nn_amd.QuantizedMLP(*q, nn_amd.QuantType.Q4_K, hidden, inter)
    g, u, d = (make_weight("q4_k", b, *s) for b, s in zip(q, ((inter, hidden), (inter, hidden), (hidden, inter))))
    x = torch.from_numpy(nn_amd.synth_normal(5, 4, (m, hidden), 1.0)).to(dev).to(xdt)
    y = mlp.forward(x)
    gate, up = nn_amd.quantized_linear(x, g).double(), nn_amd.quantized_linear(x, u).double()
    ref = (gate * torch.sigmoid(gate) * up) @ d.dequantize().double().t()
    assert (y.double() - ref).abs().max().item() <= 1e-5 * ref.pow(2).mean().sqrt().item()
    x[11, 3] = float("nan")
    z = mlp.forward(x, check=False)
    keep = torch.arange(m) != 11
    assert torch.equal(z[keep], y[keep]) and torch.isnan(z[11]).all()
    with pytest.raises(nn_amd.NonFiniteData):
        mlp.forward(x)
