"""Scratch memory (register spills) of every kernel of the built library, from the metadata of its code objects.  A spill inside
a main loop costs more than what it was meant to save (four-block fp16 tiles with zero points and kept constants: 19 registers,
7-18 % slower), and neither a build nor a numerics test shows it.  The kernels listed here have always had theirs."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"
# bytes of scratch per lane, by demangled template arguments
SPILLS = {
    # DT, MB, ZP, GM, BITS, ZPF, FP8, FP4, NW (GM 2: per-row scale lookup; MB 1, GM 0: groups of 32 and others the decode kernel lacks)
    "skinny_kernel<0, 1, true, 0, 4, false, false, 0, 4>": 100,
    "skinny_kernel<0, 1, true, 0, 4, false, false, 0, 8>": 100,
    "skinny_kernel<1, 1, false, 0, 4, false, false, 0, 4>": 24,
    "skinny_kernel<1, 1, false, 0, 4, false, false, 0, 8>": 24,
    "skinny_kernel<1, 1, true, 0, 4, false, false, 0, 4>": 96,
    "skinny_kernel<1, 1, true, 0, 4, false, false, 0, 8>": 96,
    "skinny_kernel<0, 4, false, 2, 4, false, false, 0, 8>": 24,
    "skinny_kernel<0, 4, false, 2, 8, false, false, 0, 8>": 92,
    "skinny_kernel<1, 4, false, 2, 4, false, false, 0, 8>": 64,
    "skinny_kernel<1, 4, false, 2, 8, false, false, 0, 8>": 116,
    # DT, ZP, CHANNEL, MOE, FP4, BITS, FP8, ZPF: 8-bit weights
    "mid_kernel<0, false, false, false, 0, 8, false, false>": 48,
    "mid_kernel<0, false, false, false, 0, 8, true, false>": 12,
    "mid_kernel<0, false, false, true, 0, 8, false, false>": 16,
    "mid_kernel<0, false, false, true, 0, 8, true, false>": 8,
    "mid_kernel<1, false, false, false, 0, 8, false, false>": 12,
    "mid_kernel<1, false, false, false, 0, 8, true, false>": 12,
    "mid_kernel<1, false, false, true, 0, 8, false, false>": 8,
    "mid_kernel<1, false, false, true, 0, 8, true, false>": 8,
}


def _code_objects(blob):
    """The gfx950 code objects of an (uncompressed) offload section: one bundle per translation unit."""
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", blob, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            if b"gfx950" in blob[pos + 24:pos + 24 + length]:
                yield blob[at + offset:at + offset + size]
            pos += 24 + length
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", pos)


@pytest.mark.skipif(not (os.path.exists(LLVM + "/llvm-readelf") and os.path.exists(LLVM + "/llvm-objcopy") and shutil.which("c++filt")),
                    reason="no tools to read code objects with")
def test_no_kernel_spills_more_than_listed(tmp_path):
    from vllm_amd import build
    fat = tmp_path / "fat.bin"
    lib = shutil.copy(build.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([LLVM + "/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", lib, str(tmp_path / "out.so")], check=True)
    scratch = {}
    for i, code in enumerate(_code_objects(fat.read_bytes())):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        notes = subprocess.run([LLVM + "/llvm-readelf", "--notes", str(path)], check=True, capture_output=True, text=True).stdout
        names = re.findall(r"\.name: +(_Z\S+)", notes)
        sizes = re.findall(r"\.private_segment_fixed_size: +(\d+)", notes)
        assert len(names) == len(sizes)
        scratch.update(zip(names, map(int, sizes)))
    assert len(scratch) > 300  # the scan sees the kernels
    plain = subprocess.run(["c++filt"], input="\n".join(scratch), check=True, capture_output=True, text=True).stdout.split("\n")
    over = {}
    for name, size in zip(plain, scratch.values()):
        name = re.sub(r"^void |w4a16::|\(.*$", "", name)
        if size > SPILLS.get(name, 0):
            over[name] = size
    assert not over
