"""The fp32 forward's tiles (dcn2_forward_tiles.hip) at their edges, against the
oracle: every tile of the launch rule, tiles that span images, rows and pixels
that end inside a tile, K walks that do not fill a split step, a group of several
channel chunks, a channels_last output and weight groups."""
import pytest
import torch

from dcnv2_amd import _C
from oracle import oracle

from util import check

pytestmark = pytest.mark.gpu

# (B, C, H, W, Cout, k, stride, dg, wg, nhwc): tile
SHAPES = [
    (3, 40, 65, 67, 257, 1, 1, 1, 1, False),     # 256x64, one row past a tile, 2 chunks
    (70, 33, 7, 7, 2048, 1, 1, 1, 1, False),     # 256x64, 49-pixel images, 2 chunks
    (2, 64, 129, 131, 65, 1, 1, 1, 1, False),    # 128x64, 2 chunks
    (3, 160, 61, 60, 100, 1, 1, 1, 1, True),     # 128x32, K split, 5 chunks
    (3, 96, 61, 60, 128, 3, 1, 1, 1, False),     # 128x32, K split, 27 chunks
    (5, 32, 31, 29, 127, 3, 1, 1, 1, True),      # 128x32, K split, 9 chunks
    (9, 16, 45, 43, 33, 3, 1, 2, 1, False),      # 64x64, 18 chunks
    (3, 70, 9, 5, 34, 3, 2, 1, 1, True),         # 64x32, K split, 27 chunks
    (1, 3, 4, 3, 1, 1, 1, 1, 1, False),          # 64x32, K split, 1 chunk
    (2, 16, 13, 11, 32, 5, 1, 4, 1, True),       # 64x32, K split, 100 chunks
    (2, 64, 33, 35, 256, 3, 1, 1, 2, False),     # 64x32, K split, 9 chunks, weight groups
    (3, 40, 65, 67, 257, 1, 1, 1, 1, True),      # 256x64, 2 chunks, channels_last
    (2, 64, 129, 131, 65, 1, 1, 1, 1, True),     # 128x64, 2 chunks, channels_last
    (9, 16, 45, 43, 33, 3, 1, 2, 1, True),       # 64x64, 18 chunks, channels_last
    (2, 64, 103, 101, 256, 3, 1, 1, 2, False),   # 128x64, 9 chunks, weight groups
    (2, 64, 73, 71, 512, 1, 1, 1, 2, True),      # 256x64, 1 chunk, weight groups, channels_last
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(int(v)) for v in s))
def test_forward_f32_tiles(shape):
    B, C, H, W, Cout, k, stride, dg, wg, nhwc = shape
    g = torch.Generator().manual_seed(7)
    pad, kk = k // 2, k * k
    Ho, Wo = (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1
    x = torch.randn(B, C, H, W, generator=g)
    w = torch.randn(Cout, C // wg, k, k, generator=g) * (2.0 / (C // wg * kk)) ** 0.5
    off = torch.randn(B, 2 * dg * kk, Ho, Wo, generator=g) * 1.5
    mask = torch.rand(B, dg * kk, Ho, Wo, generator=g)
    bias = torch.randn(Cout, generator=g)
    ref = oracle.dcn_forward(x, w, mask, off, bias, stride=stride, padding=pad, dilation=1,
                             deformable_groups=dg, pos_f32=True)
    xd = x.cuda()
    if nhwc:
        xd = xd.contiguous(memory_format=torch.channels_last)
    out = _C.dcn_v2_forward(xd, w.cuda(), mask.cuda(), off.cuda(), bias.cuda(), stride, stride,
                            pad, pad, 1, 1, dg)
    # 2^-24 per rounding, at most C*kk products per sum added in any order:
    # sqrt(1600) * 2^-24 * (sum of magnitudes / largest result, below 8) < 2e-5
    check("output", out, ref, 2e-5)
