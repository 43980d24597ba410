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


OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MFMA_RESULT = 12   # wait states until another instruction may touch a result of eight passes (that of a 16 x 16 x 32 product takes fewer)
VALU_RESULT = 2    # ... until an MFMA, or the lane-crossing operand of another vector instruction, may read what a vector instruction wrote
SCALAR_RESULT = 5  # ... until a memory instruction may take a scalar register that a vector instruction wrote


def _registers(operands):
    """The vector and accumulator registers named in operands: {("v", 7), ("a", 12), ...}."""
    found = set()
    for kind, one, first, last in re.findall(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])", operands):
        found.update((kind, i) for i in (range(int(one), int(one) + 1) if one else range(int(first), int(last) + 1)))
    return found


def _scalar_registers(operands):
    """The scalar registers named in operands: {7, 8, ...}."""
    found = set()
    for one, first, last in re.findall(r"\bs(?:(\d+)\b|\[(\d+):(\d+)\])", operands):
        found.update(range(int(one), int(one) + 1) if one else range(int(first), int(last) + 1))
    return found


def _hazards(listing):
    """Instructions of one kernel's listing that come too soon after an MFMA or a vector instruction whose result they touch."""
    return _look(listing)[0]


def _operand_hazards(listing):
    """Vector instructions of one kernel's listing whose result is taken too soon by the lane-crossing operand of another, or as the scalar address of a
    memory instruction: what the compiler sees to, but not in front of assembly statements."""
    return _look(listing)[1]


def _look(listing):
    code, at = [], {}
    for line in listing.splitlines():
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)", line)
        if m:
            at[int(m.group(3), 16)] = len(code)
            target = re.search(r"\+0x([0-9a-f]+)>", m.group(4))
            code.append((m.group(1), m.group(2), int(target.group(1), 16) if target else None))
    start = min(at)
    regs = [_registers(ops) for _, ops, _ in code]

    def touched_within(i, states, touches):
        """Whether ``touches(j)`` holds for an instruction j on a path of fewer than ``states`` wait states behind i."""
        todo, seen = [(i + 1, 0)], set()
        while todo:
            j, waited = todo.pop()
            if j >= len(code) or waited >= states or (j, waited) in seen:
                continue
            seen.add((j, waited))
            if touches(j):
                return True
            name, ops, target = code[j]
            waited += 1 + (int(ops) if name == "s_nop" else 0)
            if name.startswith(("s_cbranch", "s_branch")):
                todo.append((at[start + target], waited))
            if name not in ("s_branch", "s_endpgm"):
                todo.append((j + 1, waited))
        return False

    found, operands = [], []
    crossing = [_registers(ops.split(",")[1]) if re.search(r"\b(?:quad_perm|row_\w+|wave_\w+):?", ops) else set() for _, ops, _ in code]
    address = [_scalar_registers(ops) if name.startswith(("global_", "buffer_", "scratch_", "flat_")) else set() for name, ops, _ in code]
    for i, (name, ops, _) in enumerate(code):
        if not name.startswith("v_"):
            continue
        scalars = _scalar_registers(" ".join(ops.split(",")[:2 if "_co_" in name else 1]))
        if scalars and touched_within(i, SCALAR_RESULT, lambda j: scalars & address[j]):
            operands.append((i, name, ops))
        if not name.startswith(("v_mfma", "v_cmp", "v_readlane", "v_readfirstlane")) and (_registers(ops.split(",")[0]) and touched_within(
                i, VALU_RESULT, lambda j: _registers(ops.split(",")[0]) & crossing[j])):
            operands.append((i, name, ops))
        result = _registers(ops.split(",")[0])
        mfma = name.startswith("v_mfma")
        # (an MFMA may go on with the result of another as its own sum: the unit keeps these in order)
        if mfma and touched_within(i, MFMA_RESULT, lambda j: result & regs[j] and not (
                code[j][0].startswith("v_mfma") and _registers(code[j][1].split(",")[0]) == result)):
            found.append((i, name, ops))
        if not mfma and result and touched_within(i, VALU_RESULT, lambda j: code[j][0].startswith("v_mfma") and result & regs[j]):
            found.append((i, name, ops))
    return found, operands


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump is not installed")
def test_nothing_touches_a_product_before_it_is_there(tmp_path):
    """The GEMM's MFMAs are assembly statements, behind which the compiler adds no wait states: it must not put a copy of an
    accumulator there either.  Looked up in the listing of every form, along all branches."""
    import __graft_entry__
    import pika_h3_flex_amd as pk

    __graft_entry__.ensure_built()
    forms = {}
    for i, image in enumerate(_code_objects(pk._lib.LIB_PATH)):
        f = tmp_path / f"{i}.elf"
        f.write_bytes(image)
        text = subprocess.run([OBJDUMP, "-d", str(f)], check=True, capture_output=True, text=True).stdout
        for name, listing in re.findall(r"^[0-9a-f]+ <(\S*gemm_kernel\S*)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.M | re.S):
            forms[name] = _hazards(listing)
            assert listing.count("v_mfma") >= 64, name
    assert len(forms) == 5 and not {n: h[:3] for n, h in forms.items() if h}, forms


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump is not installed")
def test_no_operand_of_an_assembly_statement_is_too_young(tmp_path):
    """Multiplications that take an operand from another lane, and copies from memory to LDS whose address is scalar (some of those registers are
    kept in lanes of vector registers and come back from there), are assembly statements: the compiler puts no wait states in
    front of them.  Looked up in the listing of every kernel, along all branches."""
    import __graft_entry__
    import pika_h3_flex_amd as pk

    __graft_entry__.ensure_built()
    kernels, crossings, copies = {}, 0, 0
    for i, image in enumerate(_code_objects(pk._lib.LIB_PATH)):
        f = tmp_path / f"{i}.elf"
        f.write_bytes(image)
        text = subprocess.run([OBJDUMP, "-d", str(f)], check=True, capture_output=True, text=True).stdout
        for name, listing in re.findall(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.M | re.S):
            kernels[name] = _operand_hazards(listing)
            crossings += listing.count("row_newbcast")
            copies += listing.count("global_load_lds_dwordx4")
    assert crossings > 500 and copies > 100 and any("relay" in n for n in kernels), (crossings, copies, sorted(kernels))
    assert not {n: h[:3] for n, h in kernels.items() if h}


def test_the_look_for_young_operands_finds_what_it_looks_for():
    write = "\tv_mov_b32_e32 v9, v1           // 0000000000F0: 00\n"
    cross = "\tv_mul_f32_dpp v3, v9, v4 row_newbcast:5 row_mask:0xf bank_mask:0xf // 0000000000FC: 00\n"
    lane = "\tv_readlane_b32 s12, v40, 3    // 0000000000F0: 00\n"
    copy = "\tglobal_load_lds_dwordx4 v5, s[12:13] // 000000000108: 00\n"
    move = "\ts_mov_b32 m0, s7 // 0000000000F4: 00\n"
    assert len(_operand_hazards(write + cross)) == 1 and len(_operand_hazards(lane + move + copy)) == 1
    assert not _operand_hazards(write + "\ts_nop 1 // 0000000000F4: 00\n" + cross) and not _operand_hazards(write.replace("v9", "v4") + cross)
    assert not _operand_hazards(lane + "\ts_nop 4 // 0000000000F8: 00\n" + copy) and not _operand_hazards(lane.replace("s12", "s14") + copy)
    assert len(_operand_hazards(lane + "\ts_nop 3 // 0000000000F8: 00\n" + copy)) == 1


def test_the_look_for_products_finds_what_it_looks_for():
    mfma = "\tv_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[4:7], a[0:3]// 000000000100: 00\n"
    read = "\tv_accvgpr_read_b32 v0, a2                             // 000000000110: 00\n"
    assert len(_hazards(mfma + read)) == 1
    assert not _hazards(mfma + "\ts_nop 13                         // 000000000108: 00\n" + read)
    assert not _hazards(mfma + mfma.replace("0100", "0108")) and not _hazards(mfma + read.replace("a2", "a4"))
    assert len(_hazards(mfma + "\ts_branch 1                       // 000000000108: 00 <k+0x10>\n" + "\tv_mov_b32 v9, v1 // 00000000010C: 00\n" + read)) == 1
    assert len(_hazards("\tv_mov_b32_e32 v9, v1           // 0000000000FC: 00\n" + mfma)) == 1
