"""The persistent 2-byte forward kernels at the edges of their tiles, on batches of
many small images (each image is at least one tile, so these reach the tile counts
from which the kernels are used), against the oracle."""
import pytest
import torch

from dcnv2_amd import _C
from oracle import oracle

from util import TOL, check

pytestmark = pytest.mark.gpu

# (B, C, H, W, Cout, k, stride, dg, wg, nhwc, mask)
SHAPES = [
    # role-specialised kernel: 160 tiles or more
    (163, 16, 5, 5, 33, 3, 1, 1, 1, False, True),
    (161, 72, 4, 6, 129, 3, 1, 1, 1, True, True),
    (90, 24, 12, 13, 128, 1, 1, 3, 1, False, False),
    (54, 130, 5, 5, 600, 1, 1, 2, 1, True, True),
    (170, 128, 3, 4, 256, 3, 2, 1, 2, False, True),
    (85, 40, 11, 13, 257, 1, 1, 1, 1, False, True),
    (60, 33, 5, 4, 1100, 1, 1, 1, 1, False, True),
    (45, 64, 2, 3, 8500, 1, 1, 1, 1, True, False),   # more rows than it holds: the small tiles
    (45, 64, 2, 4, 8192, 1, 1, 1, 1, True, False),   # as many as it holds
    # resident-weight kernel (fp16): 48 tiles or more
    (50, 64, 8, 3, 129, 3, 1, 1, 1, False, True),
    (49, 5, 4, 6, 256, 3, 1, 1, 1, True, False),
    (51, 33, 9, 8, 200, 3, 1, 1, 1, False, False),
    (33, 64, 4, 4, 136, 3, 1, 1, 1, False, True),    # (from 33 tiles for NCHW)
    (32, 64, 4, 4, 136, 3, 1, 1, 1, False, True),
    (48, 64, 4, 5, 136, 3, 1, 1, 1, True, True),
    (47, 64, 4, 5, 136, 3, 1, 1, 1, True, True),
    # just below either: the small tiles
    (47, 64, 8, 3, 136, 3, 1, 1, 1, False, True),
    (159, 16, 4, 4, 64, 3, 1, 1, 1, False, True),
    # the role-specialised kernel from fewer tiles: 129; 65 up to 64 rows, 25 chunks of
    # one plane; 81 at 1x1, one chunk, more than 128 rows; 160 where it stores slowly
    (129, 40, 4, 4, 72, 3, 1, 1, 1, False, True),
    (128, 40, 4, 4, 72, 3, 1, 1, 1, False, True),
    (65, 64, 4, 4, 48, 5, 1, 1, 1, False, True),
    (64, 64, 4, 4, 48, 5, 1, 1, 1, False, True),
    (81, 33, 4, 6, 136, 1, 1, 1, 1, False, True),
    (80, 33, 4, 6, 136, 1, 1, 1, 1, False, False),
    (160, 24, 5, 3, 40, 3, 1, 1, 1, False, True),
    (159, 24, 5, 3, 40, 3, 1, 1, 1, False, True),
    (159, 24, 4, 4, 40, 3, 1, 1, 1, True, True),
    # more than 1024 rows that 16-byte pieces cannot cover: the small tiles at any number
    (130, 24, 3, 5, 1025, 1, 1, 1, 1, False, True),
    (130, 24, 3, 5, 1024, 1, 1, 1, 1, False, True),
    # 512 and 516 tiles of 128 rows x 32 pixels: those, and 256 x 64 past them
    (1, 72, 64, 128, 200, 3, 1, 1, 1, False, True),
    (1, 72, 64, 129, 200, 3, 1, 1, 1, True, True),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(int(v)) for v in s))
def test_forward_many_small_images(shape, dtype):
    B, C, H, W, Cout, k, stride, dg, wg, nhwc, with_mask = shape
    g = torch.Generator().manual_seed(3)
    pad, kk = k // 2, k * k
    Ho, Wo = (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1
    x = torch.randn(B, C, H, W, generator=g).to(dtype)
    w = (torch.randn(Cout, C // wg, k, k, generator=g) * (2.0 / (C // wg * kk)) ** 0.5).to(dtype)
    off = torch.randn(B, 2 * dg * kk, Ho, Wo, generator=g).to(dtype)
    mask = torch.rand(B, dg * kk, Ho, Wo, generator=g).to(dtype) if with_mask else None
    bias = torch.randn(Cout, generator=g).to(dtype)
    ref = oracle.dcn_forward(x, w, mask, off, bias, stride=stride, padding=pad, dilation=1,
                             deformable_groups=dg, pos_f32=True)
    xd = x.cuda()
    if nhwc:
        xd = xd.contiguous(memory_format=torch.channels_last)
    geo = (stride, stride, pad, pad, 1, 1, dg)
    out = _C.dcn_v2_forward(xd, w.cuda(), mask.cuda() if with_mask else None, off.cuda(), bias.cuda(), *geo)
    check("output", out, ref, TOL[dtype])
    if with_mask:
        logit = torch.randn(mask.shape, generator=g).to(dtype)
        refl = oracle.dcn_forward(x, w, torch.sigmoid(logit.double()), off, bias, stride=stride,
                                  padding=pad, dilation=1, deformable_groups=dg, pos_f32=True)
        om = torch.cat((off, logit), 1).cuda()
        check("output (logits)", _C.dcn_v2_forward_om(xd, w.cuda(), om, bias.cuda(), *geo), refl, TOL[dtype])
