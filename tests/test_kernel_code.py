"""What the kernels' machine code has to say and no result shows reliably: the library that
is built here, disassembled."""

import glob
import os
import re
import shutil
import subprocess

import pytest

from orion_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def code_of(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    folder = str(tmp_path_factory.mktemp("code"))
    shutil.copy(_lib.KERNELS_LIB, os.path.join(folder, "k.so"))
    subprocess.run([OBJDUMP, "--offloading", "k.so"], cwd=folder, check=True, capture_output=True)

    def instructions(kernel):
        found = []
        for path in sorted(glob.glob(os.path.join(folder, "k.so.*gfx950"))):
            text = subprocess.run([OBJDUMP, "-d", path], check=True, capture_output=True,
                                  text=True).stdout
            for part in re.split(r"\n\n(?=[0-9a-f]+ <)", text):
                if kernel in part.split("\n", 1)[0]:
                    found += [line.split("//")[0].strip() for line in part.split("\n")[1:]]
        assert found
        return found
    return instructions


def test_a_layers_row_parts_are_read_past_the_caches(code_of):
    # sixteen workgroups write 8 bytes each of a row's line and may hold the line since: each
    # of the two norms reads its rows' parts by two loads, which take none of it from a cache
    loads = [line for line in code_of("txl_layer_kernel") if "buffer_load_dwordx2" in line]
    assert sum(line.endswith(" sc1") for line in loads) == 4
    # the one other: eight bytes of a line that one workgroup has written
    assert len(loads) == 5
