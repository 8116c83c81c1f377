"""What the compiler made of the kernels, read from the built library's own metadata (no GPU)."""
import os
import re
import struct
import subprocess

from illatio_amd import hip

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def kernels(tmp_path):
    """(name, metadata text) of every kernel: the library's code objects are bundles of one ELF a source file."""
    section = tmp_path / "fatbin"
    subprocess.check_call([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", f".hip_fatbin={section}", hip.LIB_PATH, str(tmp_path / "copy.so")])
    data, out = section.read_bytes(), []
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.end() + 8
        for _ in range(struct.unpack_from("<Q", data, m.end())[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length].decode()
            at += 24 + length
            if "gfx950" not in target:
                continue
            elf = tmp_path / "elf"
            elf.write_bytes(data[m.start() + offset:m.start() + offset + size])
            notes = subprocess.check_output([os.path.join(LLVM, "llvm-readelf"), "--notes", str(elf)], text=True)
            for part in re.split(r"\n  - (?=\.agpr_count)", notes)[1:]:
                out.append((re.search(r"\n    \.name: +(\S+)", part)[1], part))
    return out


# Kernels that do, and how many registers at most: the 128 x 128 cut of the exact products keeps all 256 registers busy and leaves a
# few to scratch; the short pass's routing of more than 512 experts runs once a pass.
SPILLS = {"gemm_i8r_kernelILi0ELi4ELi4ELi1E": 4, "gemm_i8r_kernelILi12ELi4ELi4ELi1E": 4, "gemm_i8r_kernelILi14ELi4ELi4ELi1E": 4,
          "gemm_bf16_kernelILi14ELi128ELi128ELi2E": 1, "small_route_kernelILi16E": 3312}


def test_no_other_kernel_spills_its_vector_registers(tmp_path):
    found = kernels(tmp_path)
    assert len(found) > 100
    over = {}
    for name, text in found:
        n = int(re.search(r"\.vgpr_spill_count: +(\d+)", text)[1])
        if n > max([most for part, most in SPILLS.items() if part in name], default=0):
            over[name] = n
    assert not over
