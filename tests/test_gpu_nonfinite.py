"""Infinities and NaN: a sample outside the image contributes nothing whatever its
mask value or column gradient, and leaves every other result finite."""
import pytest
import torch

from dcnv2_amd import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hw", [(5, 7), (8, 8)])
def test_nonfinite_outside_samples(dtype, hw):
    H, W = hw
    B, C, Cout = 2, 64, 40
    g = torch.Generator().manual_seed(2)
    x = torch.randn(B, C, H, W, generator=g)
    w = torch.randn(Cout, C, 1, 1, generator=g) * 0.1
    off = torch.zeros(B, 2, H, W)
    mask = torch.rand(B, 1, H, W, generator=g)
    go = torch.randn(B, Cout, H, W, generator=g)
    # samples far outside, with mask values and output gradients that are not finite
    for n, (m, v) in enumerate([(float("inf"), 1.0), (float("nan"), 1.0), (0.5, float("inf")),
                                (0.5, float("nan"))]):
        off[0, :, 1, n] = 100.0
        mask[0, 0, 1, n] = m
        go[0, :, 1, n] = v
    t = [v.to(dtype).cuda() for v in (x, w, mask, off)]
    bias = torch.zeros(Cout, dtype=dtype, device="cuda")
    out = _C.dcn_v2_forward(*t, bias, 1, 1, 0, 0)
    gi, goff, gmask, gw, gb = _C.dcn_v2_backward(*t, bias, go.to(dtype).cuda(), 1, 1, 0, 0)
    assert (out[0, :, 1, :4] == 0).all()
    assert torch.isfinite(out).all()
    assert torch.isfinite(gi).all()          # nothing of those samples reaches grad_input
    assert (goff[0, :, 1, 2:4] == 0).all()   # (scaled by the mask value, finite for these two)
    assert (gmask[0, 0, 1, :4] == 0).all()
    keep = torch.ones(B, 1, H, W, dtype=torch.bool)
    keep[0, 0, 1, :4] = False
    assert torch.isfinite(goff.cpu()[keep.expand(-1, 2, -1, -1)]).all()
    assert torch.isfinite(gmask.cpu()[keep]).all()
