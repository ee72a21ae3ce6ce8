"""Launch rules that count on a number of waves per SIMD: the compiled kernels leave registers for them."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flagattention_amd", "csrc")


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")
def test_dropout_kernels_hold_the_waves_their_groups_are_chosen_by():
    """Every instance, whatever its number of wave groups: four waves per SIMD at head_dim 64, three at 128 (drop_groups and
    the order of the workgroups both assume them resident)."""
    run = subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang",
                          "-target-feature", "-Xclang", "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "-c",
                          "--cuda-device-only", "-o", os.devnull, os.path.join(CSRC, "flash_dropout.hip")],
                         check=True, capture_output=True, text=True, timeout=600)
    waves = re.findall(r"Function Name: \S*flash_dropout_fwd_kernelILi(\d+)E\S*Li(\d)ELb([01])EE.*?Occupancy \[waves/SIMD\]: (\d+)", run.stderr, re.S)
    assert {(int(d), int(groups), int(wide)) for d, groups, wide, _ in waves} == {
        (64, 1, 0), (64, 2, 0), (64, 4, 0), (64, 1, 1), (128, 1, 0), (128, 2, 0), (128, 1, 1)}
    for d, groups, wide, n in waves:
        assert int(n) >= (4 if d == "64" else 3), (d, groups, wide, n)
