"""The fp32 backward's GEMM kernels (dcn2_backward_f32.hip) at the edges of their
tiles, against the oracle: pixel tiles that span images and end early, rows that
end inside a step, one and several channel tiles per group, both layouts of
grad_output, weight groups."""
import pytest
import torch

from dcnv2_amd import _C
from oracle import oracle

from util import GRADS, TOL, check

pytestmark = pytest.mark.gpu

# (B, C, H, W, Cout, k, stride, dg, wg, nhwc, logits)
SHAPES = [
    (40, 64, 7, 7, 33, 1, 1, 1, 1, False, False),    # 49-pixel images, one channel tile
    (3, 64, 131, 127, 257, 1, 1, 1, 1, False, True),  # many 64-pixel tiles, one row past a step
    (9, 200, 14, 14, 65, 1, 1, 1, 1, False, True),   # 224 padded channels: seven 32-channel tiles share the corner sums
    (2, 256, 13, 9, 31, 3, 1, 2, 1, True, False),    # two tiles per group, channels_last
    (3, 96, 11, 10, 130, 3, 2, 1, 1, False, False),  # 96 padded channels: three 32-channel tiles
    (1, 3, 3, 4, 1, 1, 1, 1, 1, False, True),        # the smallest
    (2, 20, 9, 30, 64, 5, 1, 4, 1, True, True),      # 32-channel groups of 5 channels
    (2, 128, 17, 15, 256, 3, 1, 1, 2, False, False),  # weight groups: each tile its group's rows
    (2, 64, 17, 15, 256, 3, 1, 1, 2, True, False),   # weight groups of one 32-channel chunk
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(int(v)) for v in s))
def test_backward_f32_tiles(shape):
    B, C, H, W, Cout, k, stride, dg, wg, nhwc, logits = shape
    g = torch.Generator().manual_seed(11)
    pad, kk = k // 2, k * k
    Ho, Wo = (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1
    x = torch.randn(B, C, H, W, generator=g)
    w = torch.randn(Cout, C // wg, k, k, generator=g) * (2.0 / (C // wg * kk)) ** 0.5
    off = torch.randn(B, 2 * dg * kk, Ho, Wo, generator=g) * 1.5
    logit = torch.randn(B, dg * kk, Ho, Wo, generator=g)
    mask = torch.sigmoid(logit.double()) if logits else torch.rand(logit.shape, generator=g)
    bias = torch.randn(Cout, generator=g)
    go = torch.randn(B, Cout, Ho, Wo, generator=g)
    ref = [torch.as_tensor(v) for v in
           oracle.dcn_backward(x, w, mask, off, bias, go, stride=stride, padding=pad, dilation=1,
                               deformable_groups=dg, pos_f32=True)]
    xd, god = x.cuda(), go.cuda()
    if nhwc:
        xd, god = (t.contiguous(memory_format=torch.channels_last) for t in (xd, god))
    geo = (stride, stride, pad, pad, 1, 1, dg)
    if logits:
        gi, gom, gw, gb = _C.dcn_v2_backward_om(
            xd, w.cuda(), torch.cat((off, logit), 1).cuda(), bias.cuda(), god, *geo)
        got = [gi, gom[:, :2 * dg * kk], gom[:, 2 * dg * kk:], gw, gb]
        ref[2] = ref[2] * mask * (1 - mask)
    else:
        got = _C.dcn_v2_backward(xd, w.cuda(), mask.cuda(), off.cuda(), bias.cuda(), god, *geo)
    for name, a, r in zip(GRADS, got, ref):
        # 2^-24 per rounding over at most 50000 additions in any order: a random
        # walk of 224 * 2^-24 = 1.4e-5 of a result, against the largest one
        check(name, a, r, 2e-5)


def test_channels_last_costs_no_more_than_nchw():
    """grad_bias of a channels-last grad_output: with an atomic per load in place of one
    per row and workgroup this layer took 2.2 times the time of its NCHW form (now 1.0;
    the bound leaves room for a busy machine)."""
    g = torch.Generator().manual_seed(1)
    B, C, H, W, Cout = 5, 28, 42, 86, 91
    x, go = torch.randn(B, C, H, W, generator=g).cuda(), torch.randn(B, Cout, H, W, generator=g).cuda()
    w, b = torch.randn(Cout, C, 1, 1, generator=g).cuda(), torch.randn(Cout, generator=g).cuda()
    off, mask = torch.randn(B, 4, H, W, generator=g).cuda(), torch.rand(B, 2, H, W, generator=g).cuda()

    def run(fmt):
        xs, gs = x.contiguous(memory_format=fmt), go.contiguous(memory_format=fmt)
        times = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(20):
                grads = _C.dcn_v2_backward(xs, w, mask, off, b, gs, 1, 1, 0, 0, 1, 1, 2)
            e1.record()
            e1.synchronize()
            times.append(e0.elapsed_time(e1))
        return min(times), grads[4]

    t0, gb0 = run(torch.contiguous_format)
    t1, gb1 = run(torch.channels_last)
    ref = go.double().sum((0, 2, 3)).cpu()
    check("grad_bias", gb0, ref, TOL[torch.float32])
    check("grad_bias (channels_last)", gb1, ref, TOL[torch.float32])
    assert t1 < 1.6 * t0


def test_bias_costs_little():
    """grad_bias of odd maps (4-byte grad_output loads): with two rows to an atomic
    instruction this layer's backward took 1.9 times its time without bias (now 1.03)."""
    g = torch.Generator().manual_seed(1)
    B, C, H, W, Cout = 2, 11, 151, 105, 64
    x, go = torch.randn(B, C, H, W, generator=g).cuda(), torch.randn(B, Cout, H, W, generator=g).cuda()
    w, bias = torch.randn(Cout, C, 1, 1, generator=g).cuda(), torch.randn(Cout, generator=g).cuda()
    off, mask = torch.randn(B, 2, H, W, generator=g).cuda(), torch.rand(B, 1, H, W, generator=g).cuda()

    def run(b):
        times = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(20):
                grads = _C.dcn_v2_backward(x, w, mask, off, b, go, 1, 1, 0, 0, 1, 1, 1)
            e1.record()
            e1.synchronize()
            times.append(e0.elapsed_time(e1))
        return min(times), grads[4]

    t1, gb = run(bias)
    check("grad_bias", gb, go.double().sum((0, 2, 3)).cpu(), TOL[torch.float32])
    assert t1 < 1.4 * run(None)[0]
