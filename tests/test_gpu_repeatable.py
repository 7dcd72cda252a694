"""grad_offset and grad_mask of groups whose channels several workgroups share are the
same bits in every run where the library says so: fp32, and 16-bit grad_output rows that
are copied with padding.  Three or more parts per sample (the sum of two does not
depend on their order)."""
import pytest
import torch

from dcnv2_amd import _C
from oracle import oracle
from util import TOL, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,C,H,W,Cout,k,dg,nhwc", [
    (torch.float32, 2, 512, 14, 14, 64, 1, 1, False),    # 8 tiles of 64 channels
    (torch.float32, 2, 352, 13, 17, 40, 3, 1, False),    # 11 of 32
    (torch.float32, 2, 640, 9, 11, 40, 3, 2, True),      # 5 of 64 per group
    (torch.bfloat16, 2, 256, 25, 21, 64, 3, 1, False),   # ragged rows: 4 chunks of 64
    (torch.float16, 2, 384, 25, 21, 64, 1, 2, False),    # 3 per group
    (torch.float16, 2, 256, 16, 16, 60, 3, 1, True),     # ragged channels
], ids=["f32", "f32_ct32", "f32_dg2_nhwc", "bf16_ragged", "f16_dg2_ragged", "f16_nhwc_ragged"])
def test_offset_and_mask_gradients_repeat(dtype, B, C, H, W, Cout, k, dg, nhwc):
    g = torch.Generator().manual_seed(3)
    kk = k * k
    t = [torch.randn(B, C, H, W, generator=g), torch.randn(Cout, C, k, k, generator=g) * (2.0 / (C * kk)) ** 0.5,
         torch.rand(B, dg * kk, H, W, generator=g), torch.randn(B, 2 * dg * kk, H, W, generator=g),
         torch.randn(Cout, generator=g), torch.randn(B, Cout, H, W, generator=g)]
    t = [v.to(dtype) for v in t]
    ref = oracle.dcn_backward(*t, stride=1, padding=k // 2, dilation=1, deformable_groups=dg, pos_f32=True)
    dev = [v.cuda() for v in t]
    if nhwc:
        dev[0], dev[5] = (dev[i].contiguous(memory_format=torch.channels_last) for i in (0, 5))

    def run():
        return _C.dcn_v2_backward(*dev, 1, 1, k // 2, k // 2, 1, 1, dg)[1:3]

    first = run()
    for name, got, r in zip(("grad_offset", "grad_mask"), first, ref[1:3]):
        check(name, got, r, TOL[dtype])
    for _ in range(20):
        for a, b in zip(run(), first):
            assert torch.equal(a, b)
