"""What the library's host code plans for a call, read on the CPU through
``plan_probe.cpp``: every slice of a backward call uses no more of the workspace than
its layout holds, and all slices take the same grad_input kernel; the forward kernel on
either side of the lines between them."""
import glob
import os
import subprocess

import pytest

from dcnv2_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))
DEFAULT_BUDGET = 192 << 20
F32, F16, BF16 = 0, 1, 2


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    objs = glob.glob(os.path.join(build.BUILD, "*.o"))
    if len(objs) != len([f for f in os.listdir(build.CSRC) if f.endswith((".hip", ".cpp"))]):
        build.build(verbose=False)
        objs = glob.glob(os.path.join(build.BUILD, "*.o"))
    exe = str(tmp_path_factory.mktemp("plan") / "plan_probe")
    hipcc = [build.HIPCC, f"--offload-arch={build.ARCH}"]
    for cmd in ([*hipcc, "-std=c++17", "-c", os.path.join(HERE, "plan_probe.cpp"), "-o", exe + ".o"],
                [*hipcc, "-Wl,--allow-multiple-definition", exe + ".o", *objs, "-o", exe]):
        subprocess.run(cmd, check=True, capture_output=True)

    def run(budget, push, desc):
        r = subprocess.run([exe], input=" ".join(str(v) for v in (budget, push, *desc)), text=True,
                           capture_output=True, check=True)
        rows = [[int(v) for v in ln.split()] for ln in r.stdout.splitlines() if ln]
        return rows[0], rows[1:]

    return run


def _desc(dtype, B, C, H, W, Cout, k, dg=1, wg=1, nhwc=0):
    return (B, C, H, W, Cout, k, k, 1, 1, k // 2, k // 2, 1, 1, dg, dtype, wg, nhwc, nhwc)


# The last slice is shorter than the others, so that it alone has fewer than 128
# (bucket, channel chunk) pairs, the count from which grad_input goes by cells; each
# bucket of its interior holds more than one batch (4096) of samples.
@pytest.mark.parametrize("case,slices,pairs", [
    ((F16, 7, 128, 63, 63, 128, 5), (4, 3), 32),      # 4 images by cells: 128 pairs
    ((F16, 5, 64, 104, 104, 64, 5), (3, 2), 49),      # 147
    ((F32, 7, 128, 63, 63, 64, 5), (3, 3, 1), 64),    # 192
    ((F16, 11, 64, 47, 47, 64, 7, 2), (4, 4, 3), 18), # 72: by pixels throughout
], ids=str)
def test_short_last_slice_keeps_the_kernel(probe, case, slices, pairs):
    _, got = probe(DEFAULT_BUDGET, -1, _desc(*case))
    assert tuple(r[0] for r in got) == slices
    assert {r[1] for r in got} == {int(slices[0] * pairs >= 128)}
    for r in got:
        for need, room in zip(r[2::2], r[3::2]):
            assert need <= room


def test_slices_fit_their_layout(probe):
    """The same over batches, budgets and both forced kernels."""
    for case in ((F16, 64, 63, 63, 128, 5), (F16, 128, 63, 63, 300, 5), (F32, 96, 40, 90, 64, 7),
                 (F16, 192, 33, 20, 64, 3), (F32, 512, 14, 14, 64, 1)):
        for B in range(1, 24, 2):
            for budget in (16 << 20, 100 << 20, DEFAULT_BUDGET):
                for push in (-1, 0, 1):
                    _, got = probe(budget, push, _desc(case[0], B, *case[1:]))
                    assert sum(r[0] for r in got) == B and len({r[1] for r in got}) == 1
                    assert push < 0 or got[0][1] == push
                    for r in got:
                        assert all(need <= room for need, room in zip(r[2::2], r[3::2]))


# The lines as measured (see forward_few_tiles): tiles of 128 pixels x 256 rows (128 up to
# 128 rows), one image of 16 pixels a row (15 where rows are ragged) to a tile.
@pytest.mark.parametrize("C,Cout,k,nhwc,ragged,dg,wg,most", [
    (128, 256, 3, 0, False, 1, 1, 128), (128, 128, 7, 0, False, 1, 1, 128), (64, 512, 3, 0, False, 1, 1, 64),
    (256, 256, 5, 1, False, 1, 1, 128), (128, 100, 3, 1, False, 1, 1, 159), (64, 256, 1, 1, False, 1, 1, 159),
    (64, 64, 1, 0, False, 1, 1, 159), (64, 64, 3, 0, False, 1, 1, 128), (64, 64, 5, 0, False, 1, 1, 64),
    (64, 40, 7, 1, False, 1, 1, 64), (128, 64, 7, 0, False, 1, 1, 128), (64, 256, 1, 0, False, 1, 1, 80),
    (65, 256, 1, 0, False, 1, 1, 128), (64, 256, 5, 0, True, 1, 1, 159), (64, 64, 7, 0, True, 1, 1, 128),
    (256, 256, 3, 0, False, 1, 2, 128), (36, 446, 5, 0, True, 4, 1, 64),
    (36, 5, 7, 1, False, 4, 1, 64), (36, 40, 3, 0, False, 4, 1, 64), (36, 72, 3, 1, False, 2, 1, 128),
])
def test_few_tiles_of_the_16_bit_forward(probe, C, Cout, k, nhwc, ragged, dg, wg, most):
    for dtype in (F16, BF16):
        for B in (most, most + 1):
            _, few, _ = probe(DEFAULT_BUDGET, -1, _desc(dtype, B, C, 7, 15 if ragged else 16, Cout, k,
                                                        dg=dg, wg=wg, nhwc=nhwc))[0]
            assert few == (B == most)


def test_wide_ragged_layers_take_the_small_tiles(probe):
    for Cout, ragged, nhwc, few in ((1024, 1, 0, 0), (1028, 1, 0, 1), (1032, 0, 0, 0), (1028, 0, 1, 1), (1032, 1, 1, 0)):
        assert probe(DEFAULT_BUDGET, -1, _desc(F16, 200, 64, 7, 15 if ragged else 16, Cout, 1, nhwc=nhwc))[0][1] == few


def test_few_tiles_of_the_resident_weight_forward(probe):
    for nhwc, most in ((0, 32), (1, 47)):
        for B in (most, most + 1):
            rw, few, _ = probe(DEFAULT_BUDGET, -1, _desc(F16, B, 64, 8, 16, 256, 3, nhwc=nhwc))[0]
            assert rw == (B > most) and few == 1


def test_padded_grad_output(probe):
    def pad(*a, **kw):
        return probe(DEFAULT_BUDGET, -1, _desc(*a, **kw))[0][2]

    assert not pad(F32, 2, 64, 9, 9, 64, 1) and not pad(F16, 2, 64, 8, 9, 60, 1)  # fp32; N % 8 == 0
    assert pad(F16, 1, 64, 9, 9, 512, 1) and not pad(F16, 1, 64, 9, 9, 513, 1)   # one chunk of K
    assert pad(F16, 1, 65, 9, 9, 513, 1) and pad(F16, 1, 64, 9, 9, 513, 3)       # more
    assert not pad(BF16, 95, 64, 9, 9, 513, 1) and pad(BF16, 96, 64, 9, 9, 513, 1)  # tiles of 128 pixels
    assert pad(F16, 1, 64, 9, 9, 513, 1, nhwc=1) and not pad(F16, 1, 64, 9, 9, 520, 1, nhwc=1)
