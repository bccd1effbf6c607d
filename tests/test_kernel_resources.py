"""What the compiler gives the hot kernels (CPU only: the device code is cross-compiled).

A register that does not fit goes to scratch memory, a round trip for each use
in a kernel that is one chain of round trips, and its time follows.
"""
import os
import re
import subprocess

import pytest

from streamgc_amd import build

KERNELS = ["k_apply_elem", "k_apply_quads", "k_apply_seg"]


@pytest.fixture(scope="module")
def resources(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "kernels.s"
    subprocess.run([build._hipcc(), f"--offload-arch={build.ARCH}", *build.COMMON, *build.DEVICE,
                    "--offload-device-only", "-S", os.path.join(build.CSRC, "sgc_kernels.hip"), "-o", str(out)],
                   check=True, stderr=subprocess.DEVNULL)
    found = {}
    for entry in re.split(r"\n  - \.a", out.read_text().split("amdhsa.kernels:")[1]):
        name = re.search(r"\.name:\s*(\S+)", entry)
        if name:
            found[name.group(1)] = {k: int(v) for k, v in re.findall(r"\.(\w+):\s+(\d+)\n", entry)}
    return found


@pytest.mark.parametrize("kernel", KERNELS)
def test_per_update_kernels_use_no_scratch(kernel, resources):
    mine = {n: r for n, r in resources.items() if kernel in n}
    assert mine
    for name, r in mine.items():
        assert r["private_segment_fixed_size"] == 0 and r["vgpr_spill_count"] == 0, (name, r)
        assert r["vgpr_count"] <= 168, (name, r)   # three wavefronts a SIMD


def test_full_sweeps_fill_the_chip(resources):
    """Sweeps with a wavefront for every row: 8 wavefronts a SIMD, whatever the other variants take."""
    mine = {n: r for n, r in resources.items() if re.search(r"k_(compact|tier1_elem)ILb1E", n)}
    assert len(mine) == 2
    for name, r in mine.items():
        assert r["private_segment_fixed_size"] == 0 and r["vgpr_count"] <= 64, (name, r)
