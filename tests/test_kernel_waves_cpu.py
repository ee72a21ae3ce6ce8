"""Launch rules that count on a number of waves per SIMD: the compiled kernels leave registers for them."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flagattention_amd", "csrc")


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")
def test_dropout_kernels_hold_the_waves_their_groups_are_chosen_by():
    """Every instance, whatever its number of wave groups: four waves per SIMD at head_dim 64, two at 128 (drop_groups and
    the order of the workgroups both assume them resident)."""
    run = subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang",
                          "-target-feature", "-Xclang", "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "-c",
                          "--cuda-device-only", "-o", os.devnull, os.path.join(CSRC, "flash_dropout.hip")],
                         check=True, capture_output=True, text=True, timeout=600)
    waves = re.findall(r"Function Name: \S*flash_dropout_fwd_kernelILi(\d+)E\S*Li(\d)EE.*?Occupancy \[waves/SIMD\]: (\d+)", run.stderr, re.S)
    assert sorted((int(d), int(groups)) for d, groups, _ in waves) == [(64, 1), (64, 1), (64, 2), (64, 2), (64, 4), (64, 4),
                                                                       (128, 1), (128, 1), (128, 2), (128, 2)]
    for d, groups, n in waves:
        assert int(n) >= (4 if d == "64" else 2), (d, groups, n)
