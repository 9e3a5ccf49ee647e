"""Kernels whose loads are written in assembly keep everything in registers.

The compiler takes the output of such a load as written when the statement is: a register it spilled while the load was in
flight would be saved as it was before.  So no instance of these kernels may use scratch memory.
"""
import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

from kiln_amd import _lib

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin") or shutil.which("llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
KERNELS = ("w4a16_decode_gmp_kernel", "w4a16_mid_kernel", "w4a16_prefill_kernel")


def device_objects(blob: bytes):
    """The gfx950 code objects of every offload bundle in a library built here."""
    at = blob.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", blob, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(min(count, 8)):
            offset, size, id_len = struct.unpack_from("<QQQ", blob, pos)
            target = blob[pos + 24 : pos + 24 + id_len]
            pos += 24 + id_len
            if target.endswith(b"gfx950") and size:
                yield blob[at + offset : at + offset + size]
        at = blob.find(MAGIC, at + 1)


@pytest.mark.skipif(READELF is None, reason="llvm-readelf is not installed")
@pytest.mark.skipif(not Path(_lib.LIB_PATH).exists(), reason="the library is not built")
def test_no_kernel_with_loads_in_flight_uses_scratch_memory(tmp_path):
    seen, bad = dict.fromkeys(KERNELS, 0), []
    for i, obj in enumerate(device_objects(Path(_lib.LIB_PATH).read_bytes())):
        path = tmp_path / f"{i}.co"
        path.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        fields = [re.findall(rf"\.{f}:\s+(\S+)", notes) for f in ("symbol", "private_segment_fixed_size", "vgpr_spill_count")]
        assert len(fields[0]) == len(fields[1]) == len(fields[2])
        for symbol, scratch, spilled in zip(*fields):
            for kernel in KERNELS:
                if kernel in symbol:
                    seen[kernel] += 1
                    if int(scratch) or int(spilled):
                        bad.append((symbol, int(scratch), int(spilled)))
    assert all(seen.values()), seen
    assert not bad, bad
