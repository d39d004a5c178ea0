"""What the compiler reports of the built kernels, where a kernel's speed rests on it."""
import os
import re
import shutil
import subprocess

import pytest

from longcat_video_amd import _capi

LLVM = "/opt/rocm/llvm/bin/"


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    if not (os.path.exists(LLVM + "llvm-objdump") and os.path.exists(LLVM + "llvm-readelf") and os.path.exists(_capi.LIB_PATH)):
        pytest.skip("needs the built library, llvm-objdump and llvm-readelf")
    where = tmp_path_factory.mktemp("objects")
    lib = shutil.copy(_capi.LIB_PATH, where)
    subprocess.run([LLVM + "llvm-objdump", "--offloading", lib], check=True, capture_output=True, cwd=where)
    return sorted(str(p) for p in where.iterdir() if p.name.endswith("gfx950"))


def metadata(code_objects, name):
    """{symbol: its entry of the AMDGPU metadata} of the kernels whose symbol holds `name`."""
    found = {}
    for obj in code_objects:
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", obj], check=True, capture_output=True, text=True).stdout
        for entry in notes.split("  - .agpr_count:")[1:]:
            symbol = re.search(r"\n    \.name: +(\S+)", entry).group(1)
            if name in symbol:
                found[symbol] = entry
    assert found, name
    return found


def number(entry, key):
    return int(re.search(r"\.%s: +(\d+)" % key, entry).group(1))


def test_the_preparation_pass_stays_in_registers(code_objects):
    """It runs at the rate of a copy; a row's values through scratch memory would be another pass."""
    for symbol, entry in metadata(code_objects, "14prepare_kernel").items():
        assert number(entry, "vgpr_spill_count") == 0 and number(entry, "private_segment_fixed_size") == 0, symbol


def asked_for_together(code_objects, symbol):
    """Offsets of the first six scalar loads of one dword that stand in a row."""
    for obj in code_objects:
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--disassemble-symbols=" + symbol, obj], check=True, capture_output=True, text=True).stdout
        run = []
        for op, offset in re.findall(r"^\t(\S+)(?: s\d+, s\[\d+:\d+\], (0x[0-9a-f]+))?", text, re.M):
            run = run + [int(offset, 16)] if op == "s_load_dword" and offset else []
            if len(run) == 6:
                return run
    return []


@pytest.mark.parametrize("name", ["15fwd_frag_kernel", "14fwd_few_kernel", "15bwd_dkdv_kernel"])
def test_every_line_of_the_arguments_is_asked_for(code_objects, name):
    """A 64-byte line of them that is left out is a wait for memory of its own; a load behind them may read past their segment."""
    for symbol, entry in metadata(code_objects, name).items():
        args = [(int(at), int(size)) for at, size, kind in re.findall(r"\.offset: +(\d+)\s+\.size: +(\d+)\s+\.value_kind: +(\S+)", entry)
                if not kind.startswith("hidden")]
        end = max(at + size for at, size in args)
        asked = asked_for_together(code_objects, symbol)
        assert asked and max(asked) + 4 <= end, (symbol, asked, end)
        assert {at // 64 for at in asked} == set(range((end + 63) // 64)), (symbol, asked, end)
