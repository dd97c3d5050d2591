"""LDS layout of the built kernels, read from the notes of the code objects in
the library (AMDGPU metadata)."""
import os
import re
import struct
import subprocess

import pytest

from gputools_amd import build as gtbuild

READELF = os.path.join(gtbuild.ROCM, "llvm", "bin", "llvm-readelf")


def _static_lds(tmp_path):
    """{kernel: bytes of static LDS} over the AMDGPU code objects in the library."""
    blob = open(gtbuild.LIB, "rb").read()
    out, at = {}, blob.find(b"\x7fELF")
    while at >= 0:
        machine, = struct.unpack_from("<H", blob, at + 18)
        if machine == 224:   # EM_AMDGPU
            shoff, = struct.unpack_from("<Q", blob, at + 40)
            size, count = struct.unpack_from("<HH", blob, at + 58)
            path = tmp_path / "code.o"
            path.write_bytes(blob[at:at + shoff + size * count])
            notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True,
                                   check=True).stdout
            lds = None
            for line in notes.splitlines():
                m = re.search(r"\.group_segment_fixed_size:\s*(\d+)", line)
                if m:
                    lds = int(m.group(1))
                m = re.search(r"\.name:\s*(_Z\w+)", line)
                if m and lds is not None:
                    out[m.group(1)] = lds
                    lds = None
        at = blob.find(b"\x7fELF", at + 4)
    return out


@pytest.mark.skipif(not os.path.exists(READELF), reason="llvm-readelf not installed")
def test_clustering_dynamic_lds_starts_at_16_bytes(tmp_path):
    """The dynamic LDS lies behind a kernel's static LDS, whose reported size
    includes the padding between them.  hclust_group_kernel reads its column
    keys there 16 bytes at a time."""
    kernels = {k: v for k, v in _static_lds(tmp_path).items() if "hclust_group_kernel" in k}
    assert len(kernels) == 10
    assert {k: v % 16 for k, v in kernels.items()} == {k: 0 for k in kernels}
