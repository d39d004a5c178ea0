"""Instructions that inline assembly issues get no wait states from the compiler: it does not look into such a statement.
Read back from the built library: a VMEM instruction that takes an address or an offset from an SGPR must stand at least five
wait states behind the VALU instruction (v_readfirstlane, v_readlane, a compare) that wrote that SGPR (CDNA3 instruction set
architecture, "Manually Inserted Wait States")."""
import os
import re
import shutil
import subprocess

import pytest

from longcat_video_amd import _capi

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT_STATES = 5
VMEM = ("global_", "buffer_", "scratch_", "flat_")


def _sgprs(operand):
    out = set()
    for lo, hi, one in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", operand):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return out


def _instructions(code_object):
    """(kernel, opcode, operands), a branch target of no interest: the walk below goes through the text upwards."""
    kernel = None
    for line in subprocess.run([OBJDUMP, "-d", code_object], check=True, capture_output=True, text=True).stdout.splitlines():
        named = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if named:
            kernel = named.group(1)
        elif line.startswith("\t"):
            op, _, rest = line.split("//")[0].strip().partition(" ")
            yield kernel, op, rest.split(",") if rest else []


def too_close(instructions):
    """VMEM instructions that read an SGPR fewer than WAIT_STATES behind the VALU instruction that wrote it."""
    found, recent = [], []              # recent: (kernel, SGPRs a VALU instruction wrote, wait states it counts for)
    for kernel, op, operands in instructions:
        if op.startswith(VMEM):
            need, states = set().union(*map(_sgprs, operands)) if operands else set(), 0
            for other, wrote, counts in reversed(recent):
                if other != kernel or states >= WAIT_STATES:
                    break
                if wrote & need:
                    found.append((kernel, op, operands, states))
                    break
                states += counts
        wrote = _sgprs(operands[0]) if op.startswith("v_") and operands else set()
        if op.startswith(("v_add_co", "v_addc_co", "v_sub_co", "v_subb_co", "v_mad_u64", "v_div_scale")) and len(operands) > 1:
            wrote |= _sgprs(operands[1])
        recent = recent[-8:] + [(kernel, wrote, int(operands[0], 0) + 1 if op == "s_nop" else 1)]
    return found


def test_the_rule():
    read = ("k", "v_readfirstlane_b32", ["s4", " v1"])
    load = ("k", "global_load_lds_dwordx4", ["v2", " s[4:5]"])
    mov = ("k", "s_mov_b32", ["m0", " s9"])
    assert too_close([read, mov, ("k", "s_nop", ["0"]), load])
    assert not too_close([read, mov, ("k", "s_nop", ["3"]), load])
    assert not too_close([("k", "v_readfirstlane_b32", ["s6", " v1"]), load])


def test_sgpr_addresses_of_the_built_library(tmp_path):
    if not (os.path.exists(OBJDUMP) and os.path.exists(_capi.LIB_PATH)):
        pytest.skip("needs the built library and llvm-objdump")
    lib = shutil.copy(_capi.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    objects = sorted(str(p) for p in tmp_path.iterdir() if p.name.endswith("gfx950"))
    assert objects
    dma, found = 0, []
    for obj in objects:
        code = list(_instructions(obj))
        dma += sum(op.startswith("global_load_lds") for _, op, _ in code)
        found += too_close(code)
    assert dma > 0                      # the library was read
    assert not found, found[:4]


# Wait states between an MFMA and an instruction that reads or writes its result: four more than its passes.
PASSES = {"32x32x16": 8, "16x16x32": 4}


def _vgprs(operand):
    out = set()
    for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", operand):
        out |= {(kind, i) for i in range(int(lo or one), int(hi or one) + 1)}
    return out


def too_early(instructions):
    """Instructions that touch the result of an MFMA before its wait states are over (another MFMA may add to it).  An instruction counts
    one, s_nop what it says, and an MFMA is issued when the passes of those before it are over.  Along the text: not across the branch of a loop."""
    found, kernel, now, pipe_free, results = [], None, 0, 0, {}
    for k, op, operands in instructions:
        if k != kernel:
            kernel, now, pipe_free, results = k, 0, 0, {}
        passes = next((p for size, p in PASSES.items() if op.startswith("v_mfma") and size in op), 0)
        now = max(now + 1, pipe_free if passes else 0)
        touched = [_vgprs(o) for o in (operands[1:3] if passes else operands)]
        for reg in set().union(*touched):
            if reg in results and now - results[reg][0] - 1 < results[reg][1]:
                found.append((k, op, operands, reg))
                break
        if passes:
            pipe_free = now + passes
            results.update((reg, (now, passes + 4)) for reg in _vgprs(operands[0]))
        if op == "s_nop":
            now += int(operands[0], 0)
        if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
            results = {}
    return found


def test_the_rule_of_products():
    small = [("k", "v_mfma_f32_16x16x32_bf16", ["v[%d:%d]" % (i, i + 3), " v[64:67]", " a[0:3]", " 0"]) for i in (0, 4, 8, 12, 16)]
    large = [("k", "v_mfma_f32_32x32x16_f16", ["v[%d:%d]" % (i, i + 15), " v[64:67]", " a[0:3]", " 0"]) for i in (0, 16, 32)]
    read = ("k", "v_max_f32_e32", ["v70", " v3", " v71"])
    assert too_early(small[:1] + [read]) and too_early(small[:2] + [read]) and not too_early(small + [read]) and not too_early(small[1:] + [read])
    assert too_early(large[:1] + [read]) and not too_early(large + [read]) and not too_early(small[:1] + [("k", "s_nop", ["7"]), read])
    assert too_early(large[:1] + [("k", "s_nop", ["10"]), read]) and not too_early(large[:1] + [("k", "s_nop", ["11"]), read])
    assert not too_early(small[:1] * 2) and too_early(small[:1] + [("k", "v_mfma_f32_16x16x32_bf16", ["a[8:11]", " v[0:3]", " a[0:3]", " 0"])])


def test_products_of_the_built_library(tmp_path):
    """The attention kernels and the backward issue products by inline assembly and read them by the distance that the text keeps."""
    if not (os.path.exists(OBJDUMP) and os.path.exists(_capi.LIB_PATH)):
        pytest.skip("needs the built library and llvm-objdump")
    lib = shutil.copy(_capi.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    products, found = 0, []
    for obj in sorted(str(p) for p in tmp_path.iterdir() if p.name.endswith("gfx950")):
        code = list(_instructions(obj))
        products += sum(op.startswith("v_mfma") for _, op, _ in code)
        found += too_early(code)
    assert products > 0                 # the library was read
    assert not found, found[:4]
