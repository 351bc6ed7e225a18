"""The merge of many rows is a chain of trips to memory, so a round's loads have to be in flight together.  The compiler
decides that: the built code is looked at."""

import os
import re
import shutil
import subprocess

import pytest

from async_llm_amd import native

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def device_code(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler here")
    folder = tmp_path_factory.mktemp("device_code")
    lib = shutil.copy(native.LIB_PATH, folder)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=folder, check=True, capture_output=True)
    return [str(f) for f in sorted(folder.iterdir()) if f.name.endswith("gfx950")]


@pytest.mark.parametrize("element", ["4BF16", "3F16", "3F32"])
def test_a_round_of_the_row_merge_is_one_trip(device_code, element):
    # two states at a time, four runs each: a pair and four floats per state and run
    name = f"_ZN2va17merge_rows_kernelINS_{element}ELi4EEEvNS_9MergeArgsEii"
    text = "".join(subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={name}", f], capture_output=True, text=True).stdout
                   for f in device_code)
    assert name in text
    before_first_wait = re.split(r"s_waitcnt[^\n]*vmcnt", text[text.index("global_load_dwordx2"):], maxsplit=1)[0]
    assert len(re.findall(r"global_load_dwordx[24]", before_first_wait)) == 16
