"""Kernels whose registers are to stay registers: what the compiler noted in the built library about their private memory."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from swifttransformer_amd.ops import library

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def private_bytes(path, tmp_path):
    """(mangled) kernel name -> bytes of private memory a lane, from the notes of every code object in the library."""
    with open(path, "rb") as f:
        blob = f.read()
    magic, sizes = b"__CLANG_OFFLOAD_BUNDLE__", {}
    at = blob.find(magic)
    while at >= 0:
        count, p = struct.unpack_from("<Q", blob, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", blob, p)
            target = blob[p + 24:p + 24 + name]
            p += 24 + name
            if size and library.ARCH.encode() in target:
                obj = tmp_path / "object"
                obj.write_bytes(blob[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
                for kernel in notes.split("  - .agpr_count")[1:]:
                    name_of = re.search(r"^    \.name: +(\S+)", kernel, re.M).group(1)
                    sizes[name_of] = int(re.search(r"\.private_segment_fixed_size: +(\d+)", kernel).group(1))
        at = blob.find(magic, at + 1)
    return sizes


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs ROCm's readelf")
def test_no_private_memory(tmp_path):
    sizes = private_bytes(library.find_built() or library.build(), tmp_path)
    for kernel, instances in (("moe_down_sum_kernel", 8), ("moe_down_few_kernel", 2), ("moe_up_few_kernel", 4), ("delta_step_kernel", 10),
                              ("gemm_f32_split_kernel", 1), ("attn_rows_kernel", 14)):
        of = {n: v for n, v in sizes.items() if kernel in n}
        assert len(of) == instances and not any(of.values()), (kernel, of)
