"""Scratch of the role-specialised forward kernel, read off the built object: it sits at
the register limit, and spills in its step cost what they cost silently (88 bytes in
place of 24 in the channels-last f16 kernel: 35.2 against 32.6 us at 3x3, C 128 -> 256,
25,600 pixels)."""
import os
import re
import subprocess

from dcnv2_amd import build

LLVM = os.path.join(os.path.dirname(os.path.dirname(build.HIPCC)), "llvm", "bin")
# bytes per lane that the times in dcn2_forward.hip were taken with
MOST = {("f16", False): 12, ("f16", True): 24, ("bf16", False): 12, ("bf16", True): 88}


def test_forward_kernel_scratch(tmp_path):
    obj = os.path.join(build.BUILD, "dcn2_forward.hip.o")
    if not os.path.exists(obj):
        build.build(verbose=False)
    fat, co = str(tmp_path / "fat"), str(tmp_path / "co")
    for cmd in (["llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, os.devnull],
                ["clang-offload-bundler", "--type=o", "--unbundle", f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}",
                 f"--input={fat}", f"--output={co}"]):
        subprocess.run([os.path.join(LLVM, cmd[0]), *cmd[1:]], check=True, capture_output=True)
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", co], check=True, capture_output=True,
                           text=True).stdout
    found = re.findall(r"\.name: +\w*dcn2_fwd_ws_kernelI(DF16b|DF16_)Li\dELi\dELb(\d)E\w*\n"
                       r"\s+\.private_segment_fixed_size: (\d+)", notes)
    assert len(found) == 24
    for dtype, nhwc, scratch in found:
        assert int(scratch) <= MOST["bf16" if dtype == "DF16b" else "f16", nhwc == "1"]
