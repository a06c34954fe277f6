"""Registers of the built kernels, from the code objects in the library (no GPU needed)."""

import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, 'stim_amd', 'libstim_amd.so')
READELF = '/opt/rocm/llvm/bin/llvm-readelf'
MAGIC = b'__CLANG_OFFLOAD_BUNDLE__'


def _kernels(tmp_path):
    """Kernel symbol -> bytes of scratch a lane, over the library's gfx950 code objects."""
    with open(LIB, 'rb') as f:
        data = f.read()
    found = {}
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from('<Q', data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name_size = struct.unpack_from('<QQQ', data, entry)
            name = data[entry + 24:entry + 24 + name_size].decode()
            entry += 24 + name_size
            if 'gfx950' not in name or not size:
                continue
            path = tmp_path / 'code_object'
            path.write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([READELF, '--notes', str(path)], capture_output=True, text=True, check=True).stdout
            names = re.findall(r'^\s*\.name:\s+(_Z\S+)', notes, re.M)
            scratch = re.findall(r'^\s*\.private_segment_fixed_size:\s+(\d+)', notes, re.M)
            assert len(names) == len(scratch)
            found.update(zip(names, map(int, scratch)))
        at = data.find(MAGIC, at + 1)
    return found


def test_scan_kernels_use_no_scratch(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip('needs the built library and llvm-readelf')
    scans = {name: size for name, size in _kernels(tmp_path).items() if 'sym_scan' in name or 'sym_batch_kernel' in name}
    assert any('sym_batch_kernel' in name for name in scans) and any('sym_scan_fast' in name for name in scans)
    assert not any(scans.values()), scans
