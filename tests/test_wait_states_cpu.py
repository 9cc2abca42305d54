"""Wait states that the hardware does not insert: where instructions are written out, nobody but the writer does."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from mongoose_amd.build import LIB

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _kernels(tmp_path):
    """(kernel, its instructions) of the built library's device code."""
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and llvm-objdump")
    shutil.copy(LIB, tmp_path / "lib.so")                  # (the code objects are written beside it)
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    for path in sorted(glob.glob(str(tmp_path / "lib.so.*gfx950"))):
        p = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", path], stdout=subprocess.PIPE, text=True)
        name, code = None, []
        for line in p.stdout:
            if line.endswith(">:\n"):
                if name:
                    yield name, code
                name, code = line.split("<")[-1][:-3], []
            elif name and line.split("//")[0].strip():
                code.append(line.split("//")[0].strip())
        if name:
            yield name, code
        assert p.wait() == 0


def test_a_load_into_lds_is_not_the_instruction_behind_a_write_of_m0(tmp_path):
    """Between a scalar write of M0 and a load into LDS, whose target it is, the ISA asks for one wait state."""
    loads, bad = 0, []
    for name, code in _kernels(tmp_path):
        for before, at in zip([""] + code, code):
            if "_load_lds_" in at or re.match(r"buffer_load.*\blds\b", at):
                loads += 1
                if re.match(r"s_\w+ m0\b", before):
                    bad.append("%s: %s; %s" % (name, before, at))
    assert loads > 100 and not bad, bad[:5]
