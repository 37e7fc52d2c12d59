"""What the assembler makes of the copies into LDS (fprt::fill_lds), whose instructions the compiler does not see inside their inline
assembly and so does not keep apart from what comes before them: read from the disassembly of the library that is built here."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "flash-pop_amd", "flash_pop_amd", "libflashpop_hip.so")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")

# Wait states that the hardware needs, and does not insert, between a write and a buffer instruction that reads it
VALU_TO_DESCRIPTOR = 5   # a scalar register written by a vector instruction
SCALAR_TO_M0 = 1         # m0 written by a scalar instruction, where the copy's place in LDS comes from it


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: its instructions, (name, operands)}"""
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no disassembler")
    if not os.path.exists(LIBRARY):
        import __graft_entry__
        __graft_entry__.build()
    at = tmp_path_factory.mktemp("device_code")
    bundle, code = str(at / "bundle"), str(at / "code.o")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), f"--dump-section=.hip_fatbin={bundle}", LIBRARY, str(at / "copy.so")], check=True)
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", f"--input={bundle}", f"--output={code}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", "--no-leading-addr", code], check=True,
                          capture_output=True, text=True).stdout
    found = {}
    for line in text.splitlines():
        if label := re.match(r"<(\w+)>:$", line):
            body = found.setdefault(label[1], [])
        elif line.startswith("\t"):
            name, _, operands = line.split("//")[0].strip().partition(" ")
            body.append((name, [o.strip() for o in operands.split(",")]))
    return found


def scalars(operand):
    """The numbers of the scalar registers s<n> or s[<first>:<last>]."""
    if one := re.fullmatch(r"s(\d+)", operand):
        return {int(one[1])}
    if many := re.fullmatch(r"s\[(\d+):(\d+)\]", operand):
        return set(range(int(many[1]), int(many[2]) + 1))
    return set()


def too_early(body):
    """Copies into LDS, and those of them that follow too soon after a write of what they read, in the order of the instructions."""
    copies, early = 0, []
    for i, (name, operands) in enumerate(body):
        if not (name.startswith("buffer_load") and operands[-1].split()[-1] == "lds"):
            continue
        copies += 1
        descriptor, waited = scalars(operands[1]), 0
        assert len(descriptor) == 4
        for before, its in reversed(body[max(0, i - VALU_TO_DESCRIPTOR):i]):
            if before == "s_nop":
                waited += int(its[0]) + 1
                continue
            if waited < VALU_TO_DESCRIPTOR and before.startswith("v_") and scalars(its[0]) & descriptor:
                early.append((i, before, its, operands))
            if waited < SCALAR_TO_M0 and before.startswith("s_") and its[0] == "m0":
                early.append((i, before, its, operands))
            waited += 1
    return copies, early


def test_copies_into_lds_wait_for_what_they_read(kernels):
    copying = {}
    for kernel, body in kernels.items():
        copies, early = too_early(body)
        assert not early, (kernel, early[:4])
        if copies:
            copying[kernel] = copies
    assert any("retention_pass_fill_kernel" in k for k in copying) and any("retention_pass_wide_kernel" in k for k in copying), copying


def test_the_scan_sees_what_it_looks_for():
    copy = ("buffer_load_dwordx4", ["v1", "s[8:11]", "0 offen lds"])
    write, mov, other = ("v_readfirstlane_b32", ["s8", "v2"]), ("s_mov_b32", ["m0", "s4"]), ("s_add_u32", ["s1", "s2", "s3"])
    assert too_early([write, mov, ("s_nop", ["0"]), copy]) == (1, [(3, *write, copy[1])])
    assert too_early([write, other, mov, ("s_nop", ["0"]), other, copy])[1]       # four
    assert not too_early([write, mov, ("s_nop", ["3"]), copy])[1]                 # five
    assert not too_early([("v_readfirstlane_b32", ["s7", "v2"]), mov, ("s_nop", ["0"]), copy])[1]
    assert too_early([mov, copy])[1] and not too_early([mov, other, copy])[1]
