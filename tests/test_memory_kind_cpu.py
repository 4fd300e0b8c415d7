"""Where the greedy hand-off's parts may meet through device atomics: only in
the memory of the device that runs it (memory_kind.hpp, compiled for the host)."""
import shutil
import subprocess

import pytest

from ornith_g256 import _build

PROGRAM = """
#include "memory_kind.hpp"
#include <cstdio>
int main() {
    hipPointerAttribute_t own{};
    own.type = hipMemoryTypeDevice;
    own.device = 1;
    hipPointerAttribute_t managed = own, host = own, unknown = own;
    managed.isManaged = 1;
    host.type = hipMemoryTypeHost;
    unknown.type = hipMemoryTypeUnregistered;
    std::printf("%d %d %d %d %d\\n", ornith::device_atomics_reach(own, 1), ornith::device_atomics_reach(own, 0),
                ornith::device_atomics_reach(managed, 1), ornith::device_atomics_reach(host, 1),
                ornith::device_atomics_reach(unknown, 1));
}
"""


@pytest.mark.skipif(not shutil.which('g++'), reason='no g++')
def test_only_the_running_devices_own_memory(tmp_path):
    src, exe = tmp_path / 'kind.cpp', tmp_path / 'kind'
    src.write_text(PROGRAM)
    subprocess.run(['g++', '-std=c++20', '-D__HIP_PLATFORM_AMD__', '-I/opt/rocm/include', f'-I{_build.CSRC}',
                    str(src), '-o', str(exe)], check=True, capture_output=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True).stdout.split() == ['1', '0', '0', '0', '0']
