"""Register counts that keep two workgroups on a CU, read from the built library's kernel
metadata: the per-item work-queue kernels over fp8 K/V run eight waves per workgroup, so two
workgroups need at most 128 of a SIMD's 512 registers per wave."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "persistentkv-attention_amd", "libpkv.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
AMDGPU = 224  # e_machine of the code objects inside the library


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """{mangled kernel name: vector registers}"""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    assert os.path.exists(LIB), "build first"
    with open(LIB, "rb") as f:
        data = f.read()
    found, at = {}, data.find(b"\x7fELF", 1)
    while at > 0:
        if struct.unpack_from("<H", data, at + 18)[0] == AMDGPU:
            path = tmp_path_factory.mktemp("co") / "code.elf"
            path.write_bytes(data[at:])
            notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True).stdout
            for kernel in notes.split(".agpr_count:")[1:]:
                name = re.search(r"\.name:\s+(_Z\S+)", kernel)
                count = re.search(r"\.vgpr_count:\s+(\d+)", kernel)
                if name and count:
                    found[name.group(1)] = int(count.group(1))
        at = data.find(b"\x7fELF", at + 4)
    assert found
    return found


@pytest.mark.parametrize("elem", ["4Half", "6BFloat"])
def test_two_workgroups_of_fp8_queue_items_per_cu(registers, elem):
    # decode_kernel<elem, 1 head block, fp8 pager, work queue, 8 waves, ...>, fused merge or not
    ours = {n: r for n, r in registers.items()
            if n.startswith(f"_ZN3pkv13decode_kernelINS_{elem}ELi1ELi3ELi2ELi8E")}
    assert len(ours) == 4, sorted(ours)
    assert max(ours.values()) <= 128, ours
