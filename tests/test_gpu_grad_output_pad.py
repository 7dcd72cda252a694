"""Backward from the padded copy of a 2-byte grad_output (rows that 16-byte loads
cannot read): every remainder of Ho*Wo (NCHW) and of Cout (channels_last) by 8, on
the fused and the two-kernel path, more than 256 output channels, image slices, and
a misaligned grad_output; all five gradients against the oracle."""
import pytest
import torch

from dcnv2_amd import _C
from oracle import oracle

from util import GRADS, TOL, check

pytestmark = pytest.mark.gpu

# (B, C, H, W, Cout, k, dg, nhwc grad_output, slices)
SHAPES = [(2, 64, 1, n, 40, 1, 1, False, False) for n in range(1, 8)] + \
    [(2, 24, 5, 7, 24 + n, 3, 1, True, False) for n in range(1, 8)] + [
        (3, 128, 13, 11, 256, 3, 2, False, False),
        (2, 80, 9, 9, 129, 3, 1, True, False),
        (2, 64, 7, 9, 300, 3, 1, False, False),
        (2, 64, 7, 9, 301, 1, 1, True, False),
        (5, 64, 15, 17, 72, 3, 1, False, True),
        (5, 64, 15, 17, 70, 3, 1, True, True),
        # more than 512 rows and one chunk: read in place below 96 tiles of 128 pixels,
        # in slices too
        (3, 40, 5, 7, 514, 1, 1, False, False),
        (96, 8, 3, 3, 514, 1, 1, False, True),
    ]


@pytest.mark.parametrize("fused", [-1, 0])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(int(v)) for v in s))
def test_padded_grad_output(shape, dtype, fused):
    B, C, H, W, Cout, k, dg, nhwc, slices = shape
    g = torch.Generator().manual_seed(17)
    pad, kk = k // 2, k * k
    x = torch.randn(B, C, H, W, generator=g).to(dtype)
    w = (torch.randn(Cout, C, k, k, generator=g) * (2.0 / (C * kk)) ** 0.5).to(dtype)
    off = torch.randn(B, 2 * dg * kk, H, W, generator=g).to(dtype)
    mask = torch.rand(B, dg * kk, H, W, generator=g).to(dtype)
    bias = torch.randn(Cout, generator=g).to(dtype)
    go = torch.randn(B, Cout, H, W, generator=g).to(dtype)
    ref = oracle.dcn_backward(x, w, mask, off, bias, go, stride=1, padding=pad, dilation=1,
                              deformable_groups=dg, pos_f32=True)
    # one element past an aligned start: no row of it is aligned either
    god = torch.empty(go.numel() + 1, dtype=dtype, device="cuda")[1:].view(go.shape)
    god.copy_(go.cuda())
    if nhwc:
        god = god.contiguous(memory_format=torch.channels_last)
    args = [t.cuda() for t in (x, w, mask, off, bias)]
    with _C.option("bwd_fused", fused), \
            _C.option("bwd_slice_bytes", 1 if slices else _C.get_option("bwd_slice_bytes")):
        got = _C.dcn_v2_backward(*args, god, 1, 1, pad, pad, 1, 1, dg)
    for name, a, r in zip(GRADS, got, ref):
        check(name, a, r, TOL[dtype])
