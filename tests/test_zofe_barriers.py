"""The generated gfx950 code of the ZOFE column kernels keeps a barrier between
the site lists' stores and their first reads, which other wavefronts make (no
device: cross-compiled)."""
import os
import re
import subprocess

import pytest

from qspectra_amd.csrc import build as B
from tests.conftest import ROOT


def test_site_lists_are_complete_before_they_are_read(tmp_path):
    if not os.path.exists(B.hipcc()):
        pytest.skip('no hipcc')
    out = str(tmp_path / 'zofe.s')
    subprocess.run([B.hipcc(), '--offload-arch=gfx950', '-O3', '-std=c++17', '-Xclang',
                    '-target-feature', '-Xclang', '-packed-fp32-ops', '--offload-device-only',
                    '-S', '-I', os.path.join(ROOT, 'include'), '-o', out,
                    os.path.join(B.HERE, 'zofe.hip')], check=True, stderr=subprocess.DEVNULL)
    bodies = re.findall(r'^(_ZN\w*zofe_column_kernel\w*):(.*?)^\.Lfunc_end', open(out).read(),
                        flags=re.M | re.S)
    assert len(bodies) == 32                  # 8 sizes, 1 or 2 columns, with and without fields
    for name, body in bodies:
        # the lists are the kernel's only 32-bit entries in LDS
        ops = re.findall(r'\b(s_barrier|ds_write2?(?:st64)?_b32|ds_read2?(?:st64)?_b32)\b', body)
        read = next(i for i, op in enumerate(ops) if op.startswith('ds_read'))
        stores = [i for i in range(read) if ops[i].startswith('ds_write')]
        assert stores, name
        assert 's_barrier' in ops[stores[-1]:read], name
