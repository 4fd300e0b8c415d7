"""Registers of the grouped projections, as the compiler reports them: the
kernels stream codes with every register in use, and a spill puts scratch
traffic into their inner loop."""
import concurrent.futures as cf
import os
import re
import shutil
import subprocess

import pytest

from ornith_g256 import _build


def _resources(tile, out):
    cmd = [_build.HIPCC, *_build.FLAGS, f'-DORNITH_ROUTED_TILE={tile}', '--offload-device-only',
           '-Rpass-analysis=kernel-resource-usage', '-c', str(_build.CSRC / 'proj_grouped.hip'), '-o', str(out)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    kernels, name = {}, None
    for line in res.stderr.splitlines():
        m = re.search(r'Function Name: (\S+)', line)
        if m:
            name = m.group(1)
            kernels[name] = {}
        m = re.search(r'remark:.*?    (\S[^:]*): (\d+)', line)
        if m and name:
            kernels[name][m.group(1)] = int(m.group(2))
    return kernels


@pytest.mark.skipif(not (shutil.which(_build.HIPCC) or os.path.exists(_build.HIPCC)), reason='no hipcc')
def test_grouped_projections_do_not_spill(tmp_path):
    with cf.ThreadPoolExecutor(2) as pool:
        both = list(pool.map(lambda t: _resources(t, tmp_path / f'n{t}.o'), (16, 32)))
    for kernels in both:
        assert sum('gateup_tile_kernel' in k for k in kernels) >= 4
        assert sum('down_tile_kernel' in k for k in kernels) >= 4
        for name, r in kernels.items():
            assert r['VGPRs Spill'] == 0 and r['ScratchSize [bytes/lane]'] == 0, (name, r)
