"""Registers of kernels whose dispatch or residency counts on them, from the
metadata of the built library's gfx950 code objects."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")
OBJCOPY = Path("/opt/rocm/llvm/bin/llvm-objcopy")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """{mangled kernel name: (vector registers, bytes of scratch per lane)}."""
    if not (READELF.exists() and OBJCOPY.exists()):
        pytest.skip("no LLVM tools")
    from magma_amd import _ffi
    _ffi.load()
    tmp = tmp_path_factory.mktemp("code")
    fat = tmp / "fatbin"
    subprocess.run([OBJCOPY, f"--dump-section=.hip_fatbin={fat}", _ffi.LIB_PATH, tmp / "copy.so"], check=True)
    data, out, at = fat.read_bytes(), {}, 0
    while (at := data.find(MAGIC, at)) >= 0:
        p = at + len(MAGIC)
        count, = struct.unpack_from("<Q", data, p)
        p += 8
        for _ in range(count):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                elf = tmp / "code.elf"
                elf.write_bytes(data[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", elf], check=True, capture_output=True, text=True).stdout
                for rec in re.split(r"\n  - \.a", notes)[1:]:
                    n = re.search(r"\.name:\s+(\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", rec)
                    v = re.search(r"\.vgpr_count:\s+(\d+)", rec)
                    if n and v:
                        out[n.group(1)] = int(v.group(1)), int(n.group(2))
        at += len(MAGIC)
    assert out
    return out


# 512 vector registers per SIMD lane, given out in eights: 168 is the most
# that three waves can have
@pytest.mark.parametrize("kernel,most", [("getrf_tile_kernelILi5ELb0EE", 168), ("getrf_tile_kernelILi6ELb0EE", 168)])
def test_waves_per_simd(registers, kernel, most):
    found = [v for k, (v, _) in registers.items() if kernel in k]
    assert len(found) == 1 and found[0] <= most, found


def test_solve_kernels_do_not_spill(registers):
    """One register (8 bytes) at most: the solves are chains of short steps,
    and at 64..172 bytes of scratch they took up to 1.8 times as long."""
    found = {k: s for k, (_, s) in registers.items() if "getrs_" in k and "_kernel" in k}
    assert len(found) > 60 and max(found.values()) <= 8, {k: s for k, s in found.items() if s > 8}
