"""Registers of the compile-time hierarchy kernels: none keeps more than a few
values in scratch memory (no device: the compiler's resource report)."""
import os
import re
import subprocess

import pytest

from qspectra_amd.csrc import build as B
from tests.conftest import ROOT


def test_hierarchy_kernels_do_not_spill():
    """A bound on wavefronts per SIMD that one block size bears spilled 75 to
    100 registers at another (252 bytes per thread); the present ones stay at
    or below ten (36 bytes, outside the element loop's products)."""
    if not os.path.exists(B.hipcc()):
        pytest.skip('no hipcc')
    report = subprocess.run(
        [B.hipcc(), '--offload-arch=gfx950', '-O3', '-std=c++17', '-Xclang', '-target-feature',
         '-Xclang', '-packed-fp32-ops', '--offload-device-only', '-c', '-o', os.devnull,
         '-Rpass-analysis=kernel-resource-usage', '-I', os.path.join(ROOT, 'include'),
         os.path.join(B.HERE, 'heom.hip')], check=True, stderr=subprocess.PIPE,
        universal_newlines=True).stderr
    found = re.findall(r'Function Name: (\S*heom_comm_kernel\S*).*?ScratchSize[^:]*: (\d+)', report,
                       flags=re.S)
    assert len(found) == 42            # 7 sizes, 1 or 2 Matsubara terms, 3 pairs of types
    for name, scratch in found:
        assert int(scratch) <= 40, (name, scratch)
