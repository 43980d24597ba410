"""What the compiler made of the kernels: read from the code objects inside the built library, no GPU needed."""
import os
import re
import shutil
import struct
import subprocess

import pytest

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def _code_objects(path):
    """The gfx950 ELF images of a library's offload bundles (one bundle per translation unit)."""
    blob = open(path, "rb").read()
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + 24)
        pos = at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in triple and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)


@pytest.mark.skipif(not os.path.exists(READELF), reason="llvm-readelf is not installed")
def test_no_kernel_spills_registers(tmp_path):
    """Every kernel is laid out to fit its register budget; a spill inside a tile loop is scratch traffic for every key."""
    import __graft_entry__
    import pika_h3_flex_amd as pk

    __graft_entry__.ensure_built()
    spills = {}
    for i, image in enumerate(_code_objects(pk._lib.LIB_PATH)):
        f = tmp_path / f"{i}.elf"
        f.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split("- .agpr_count")[1:]:
            name = re.search(r"^\s+\.name:\s+(\S+)", kernel, re.M).group(1)
            spills[name] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel).group(1)) + int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel).group(1))
    assert any("attn_fwd_narrow_kernel" in n for n in spills) and any("gemm_kernel" in n for n in spills), sorted(spills)
    assert not {n: s for n, s in spills.items() if s}


def test_no_load_into_registers_is_inline_assembly():
    """The compiler takes the output of an assembly statement for written at once, so a load in flight could land in a register
    that holds something else by then: such loads are left to the compiler, which waits for them.  (Copies from memory
    to LDS have no register output.)"""
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pika-h3-flex_amd", "csrc")
    found = []
    for name in sorted(os.listdir(csrc)):
        if name.endswith((".hip", ".h")):
            text = open(os.path.join(csrc, name)).read()
            for m in re.finditer(r"\basm\b[^;]*;", text):
                loads = re.findall(r"\b(?:ds_read|ds_load|global_load|buffer_load|flat_load|scratch_load|s_load)_\w+", m.group(0))
                found += [(name, op) for op in loads if not op.startswith("global_load_lds")]
    assert not found
