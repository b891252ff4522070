"""The barriers of the double-buffered convolution kernels (CPU: the compiled code is read, nothing runs).

A stage's barrier lets other wavefronts load over the buffer that this one has just read, so the wait in front of
it has to name the LDS reads (lgkmcnt) beside the loads (vmcnt): nothing else orders them before the barrier.
"""
import os
import re
import subprocess
from pathlib import Path

import pytest

from tests.conftest import ROOT
from torchfdtd_amd import _native as N

HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
STAGED = ('gather_gemm_kernel', 'weight_grad_kernel')


@pytest.mark.skipif(not Path(HIPCC).exists(), reason='hipcc is not installed')
def test_every_stage_barrier_waits_for_the_lds_reads(tmp_path):
    listing = tmp_path/'conv.s'
    flags = [f for f in N.HIPCC_FLAGS if f not in ('-shared', '-fPIC')]
    subprocess.run([HIPCC, *flags, '-I', str(ROOT/'include'), '--offload-device-only', '-S', str(ROOT/'torchfdtd_amd/csrc/conv.hip'),
                    '-o', str(listing)], check=True, capture_output=True)
    kernel, wait, checked, bare = None, '', {}, []
    for line in listing.read_text().split('\n'):
        label = re.match(r'(_ZN\w+):', line)
        if label:
            kernel, wait = next((k for k in STAGED if k in label.group(1)), None), ''
        if kernel is None:
            continue
        code = line.split(';')[0].strip()
        if code.startswith('s_waitcnt'):
            wait = code
        elif code == 's_barrier':
            checked[kernel] = checked.get(kernel, 0)+1
            if 'lgkmcnt(0)' not in wait:
                bare.append((label, wait))
    assert all(checked.get(k, 0) >= 6 for k in STAGED), checked
    assert not bare, f'{len(bare)} of {sum(checked.values())} barriers wait for {sorted({w for _, w in bare})} alone'
