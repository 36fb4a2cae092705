"""GPU parity of the few-token expert kernel (at most 16 tokens and 128 assignments) against
the CPU oracle's moe_forward (crates/nn-gptoss/src/quantized_model.rs:99-194), at the edges of
its rules: one token; 16 and 17 tokens (the limit and the general path just past it); 128 and
144 assignments; every token on one expert (its rows in several items); K / 32 of 1, 16, 17,
50, 90 and 103 (more waves than k-blocks; shares of two, four, five and eight; a share past one
batch); more slots than used experts and more items than workgroups; f32 activations split in
the kernel.  Bars as tests/test_gpu_moe.py (f32 output, activations as pairs of bf16: 2^-17
relative per product, far below 1e-3)."""
import numpy as np
import pytest
import torch

from test_gpu_linear import check_close
from test_gpu_moe import make_layer, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xdt", ["bf16", "f32"])
@pytest.mark.parametrize("E,H,I,T,k,skew", [
    (1, 32, 32, 1, 1, False), (4, 32, 544, 2, 4, False), (32, 544, 64, 1, 4, False), (8, 512, 96, 16, 2, True),
    (16, 1600, 32, 16, 8, False), (16, 64, 64, 16, 9, False), (64, 96, 512, 15, 8, False), (8, 96, 96, 17, 2, True),
    (3, 64, 1600, 16, 3, False), (4, 2880, 64, 3, 2, False), (3, 64, 2880, 13, 2, False), (2, 3296, 32, 12, 2, False),
    (2, 32, 3296, 16, 2, False)])
def test_moe_few_tokens(O, E, H, I, T, k, skew, xdt):
    import nn_amd
    nn_amd.init(0)
    L = make_layer(E, H, I, seed=E * 5 + T)
    moe = upload(L, E, H, I)
    x = torch.from_numpy(nn_amd.synth_normal(23, 5, (T, H), 1.0)).cuda()
    if xdt == "bf16":
        x = x.to(torch.bfloat16)
    lg = nn_amd.synth_normal(23, 6, (T, E), 1.0)
    if skew:
        lg[:, 1] += 12.0
    y, ti, tw = moe.forward(x, torch.from_numpy(lg).cuda(), top_k=k, return_routing=True)
    ref, rti, rtw = O.moe_forward(x.float().cpu().numpy(), lg, k, L["gp"], L["gs"], L["gb"], L["dp"], L["ds"], L["db"], I)
    assert np.array_equal(ti.cpu().numpy().astype(np.uint32), rti), "routing differs"
    assert np.allclose(tw.cpu().numpy(), rtw, rtol=1e-6, atol=1e-7)
    check_close(ref, y.cpu().numpy(), f"moe few E={E} H={H} I={I} T={T} k={k} x={xdt}")


def test_moe_few_tokens_nonfinite_rows():
    """A NaN or infinity in one token stays in that token's output (rows of a tile are independent)."""
    import nn_amd
    nn_amd.init(0)
    E, H, I, T = 4, 96, 64, 5
    L = make_layer(E, H, I, seed=3)
    moe = upload(L, E, H, I)
    x = torch.from_numpy(nn_amd.synth_normal(29, 5, (T, H), 1.0)).cuda()
    lg = torch.from_numpy(nn_amd.synth_normal(29, 6, (T, E), 1.0)).cuda()
    good = moe.forward(x, lg, top_k=4)
    x[1, 7], x[3, 90] = float("nan"), float("inf")
    bad = moe.forward(x, lg, top_k=4)
    keep = [0, 2, 4]
    assert torch.equal(good[keep], bad[keep])
    assert not torch.isfinite(bad[1]).any() and not torch.isfinite(bad[3]).any()
