"""grad_input with a bucket's work shared out over workgroups (few buckets: ranges of
channel chunks and, per pixel, interleaved window passes), against the oracle on
both grad_input kernels: chunk counts that do and do not divide over the parts, one
bucket and several, a bucket of several record batches, padded channels."""
import pytest
import torch

from dcnv2_amd import _C
from oracle import oracle

from util import TOL, check

pytestmark = pytest.mark.gpu

# (B, C, H, W, k, dg, nhwc)
SHAPES = [
    (1, 64, 9, 12, 1, 1, False),     # one bucket; one chunk (16-bit) or two (fp32)
    (2, 330, 14, 14, 1, 1, False),   # 6 / 11 chunks, one bucket per image
    (1, 192, 33, 18, 3, 1, True),    # several buckets, channels_last
    (1, 160, 16, 17, 5, 2, False),   # 80 channels per group
    (1, 64, 12, 13, 7, 1, False),    # 49 taps in one bucket: several record batches
]


@pytest.mark.parametrize("by_cells", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(int(v)) for v in s))
def test_grad_input_parts(shape, dtype, by_cells):
    B, C, H, W, k, dg, nhwc = shape
    g = torch.Generator().manual_seed(5)
    pad, kk, Cout = k // 2, k * k, 40
    x = torch.randn(B, C, H, W, generator=g).to(dtype)
    w = (torch.randn(Cout, C, k, k, generator=g) * (2.0 / (C * kk)) ** 0.5).to(dtype)
    off = torch.randn(B, 2 * dg * kk, H, W, generator=g).to(dtype)
    mask = torch.rand(B, dg * kk, H, W, generator=g).to(dtype)
    bias = torch.randn(Cout, generator=g).to(dtype)
    go = torch.randn(B, Cout, H, W, generator=g).to(dtype)
    ref = oracle.dcn_backward(x, w, mask, off, bias, go, stride=1, padding=pad, dilation=1,
                              deformable_groups=dg, pos_f32=True)[0]
    xd = x.cuda()
    if nhwc:
        xd = xd.contiguous(memory_format=torch.channels_last)
    with _C.option("gi_push", by_cells):
        got = _C.dcn_v2_backward(xd, w.cuda(), mask.cuda(), off.cuda(), bias.cuda(), go.cuda(),
                                 1, 1, pad, pad, 1, 1, dg)[0]
    check("grad_input", got, ref, TOL[dtype])
