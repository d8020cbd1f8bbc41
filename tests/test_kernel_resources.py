"""Registers and waves per SIMD of kernels whose times depend on them, as the compiler reports them: no GPU needed."""
import os
import re
import subprocess

import pytest

from neus2_amd import build


def resources(source, directory):
    """The kernels of a source: mangled name -> (waves per SIMD, vector registers, spilled ones)."""
    out = subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c", os.path.join(build.CSRC, source), "-o", str(directory / "device.o")],
                         capture_output=True, text=True, check=True, timeout=300).stderr
    found = {}
    for part in out.split("Function Name: ")[1:]:
        waves, registers, spilled = (int(re.search(what + r": (\d+)", part)[1]) for what in (r"Occupancy \[waves/SIMD\]", r"\bVGPRs", "VGPRs Spill"))
        found[part.split()[0]] = waves, registers, spilled
    return found


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_the_lattices_fine_levels_have_their_waves(tmp_path):
    """One branch with more registers takes waves from all of them: six per SIMD fit 80, and what small launches have on purpose is five."""
    found = {k: v for k, v in resources("lattice.hip", tmp_path).items() if "lattice_fine_kernel" in k}
    assert sorted(v[0] for v in found.values()) == [5, 6]
    assert all(registers <= 80 and spilled == 0 for _, registers, spilled in found.values())
