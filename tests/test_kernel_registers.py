'''Registers that the compiler gave the kernels, as the built code objects state them.'''
import os
import re
import shutil
import subprocess

import pytest

from vkjax_amd.csrc import build

LLVM = '/opt/rocm/llvm/bin'


def registers(module, tmp_path):
    '''{kernel: vector registers}'''
    obj = str(tmp_path / 'code.o')
    subprocess.run([f'{LLVM}/clang-offload-bundler', '--unbundle', '--type=o', '--targets=hipv4-amdgcn-amd-amdhsa--gfx950',
                    f'--input={build.hsaco_path(module)}', f'--output={obj}'], check=True)
    notes = subprocess.run([f'{LLVM}/llvm-readelf', '--notes', obj], check=True, capture_output=True, text=True).stdout
    return {re.search(r'\.name:\s+(\S+)', k).group(1): int(re.search(r'\.vgpr_count:\s+(\d+)', k).group(1)) for k in notes.split('- .agpr_count')[1:]}


@pytest.mark.skipif(not (shutil.which(f'{LLVM}/clang-offload-bundler') and os.path.exists(build.hsaco_path('reduce'))), reason='no code object, or no tool to look into it')
def test_softmax_rows_leaves_room_for_two_waves(tmp_path):
    '''A SIMD has 512 registers: with more than 256 a kernel has a single wave there, and nothing to do while it waits for memory.'''
    counts = {k: n for k, n in registers('reduce', tmp_path).items() if k.startswith('softmax_rows')}
    assert len(counts) == 20 and max(counts.values()) <= 256, counts
