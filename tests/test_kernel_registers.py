"""Kernels whose registers are to stay registers, and few enough: what the compiler noted in the built library about their private memory
and their vector registers."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from swifttransformer_amd.ops import library

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def noted(path, tmp_path, field="private_segment_fixed_size"):
    """(mangled) kernel name -> a number that the compiler noted, from every code object in the library."""
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
                    sizes[name_of] = int(re.search(rf"\.{field}: +(\d+)", kernel).group(1))
        at = blob.find(magic, at + 1)
    return sizes


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs ROCm's readelf")
def test_no_private_memory(tmp_path):
    sizes = noted(library.find_built() or library.build(), tmp_path)
    for kernel, instances in (("moe_down_sum_kernel", 8), ("moe_down_few_kernel", 2), ("moe_up_few_kernel", 4), ("delta_step_kernel", 10),
                              ("gemm_f32_split_kernel", 1), ("attn_rows_kernel", 14), ("gemm_skinny_resident_kernel", 64),
                              ("gemm_parts_kernel", 3), ("latent_up_few_kernel", 8), ("state_out_kernel", 8)):
        of = {n: v for n, v in sizes.items() if kernel in n}
        assert len(of) == instances and not any(of.values()), (kernel, of)


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs ROCm's readelf")
@pytest.mark.parametrize("kernel,instances,most", [
    # two waves a SIMD, as many as two workgroups have in the LDS of a unit: outputs of states of more than 64 key channels (<32, 4> and <32, 8, whole pieces>)
    ("state_out_kernelILi32ELi4E", 2, 256), ("state_out_kernelILi32ELi8ELb1E", 1, 256),
    # eight: two workgroups of sixteen waves a unit
    ("gemm_skinny_resident_kernelILi16ELi1ELb0ELi0E", 2, 64), ("gemm_skinny_resident_kernelILi16ELi1ELb1ELi0E", 2, 64),
    ("gemm_skinny_resident_kernelILi16ELi2ELb0ELi3ELi8E", 1, 64), ("gemm_skinny_resident_kernelILi16ELi2ELb1ELi3ELi8E", 1, 64),
    # four: no second norm's gains
    ("rms_onto_kernelIfLi4ELi8ELb0E", 1, 128),
    # three, with some to spare: no values held beside the scores in float
    ("sink_attention_kernelIfLi1ELi4E", 1, 144)])
def test_registers_leave_room_for_another_workgroup(tmp_path, kernel, instances, most):
    counts = noted(library.find_built() or library.build(), tmp_path, "vgpr_count")
    of = {n: v for n, v in counts.items() if kernel in n}
    assert len(of) == instances and max(of.values()) <= most, (kernel, of)
