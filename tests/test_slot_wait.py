"""The slot words of the split workspace reach LDS before any wave reads them: checked on the code of the built library, the project's own kernels."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from bitladder_amd import _lib
from bitladder_amd.build import hipcc

SLOT_LOAD = "global_load_lds_dword "        # (rows go by global_load_lds_dwordx4)
BRANCH = re.compile(r"s_c?branch.*<\S+\+0x([0-9a-f]+)>")


def _kernels(tmp_path):
    """(name, [(offset, instruction, branch target or None)]) of every decode kernel in the library."""
    lib = shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    llvm = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc()))), "lib", "llvm", "bin", "llvm-objdump")
    if not os.path.exists(llvm):
        pytest.skip("no llvm-objdump")
    subprocess.run([llvm, "--offloading", lib], check=True, stdout=subprocess.DEVNULL)
    for obj in glob.glob(str(tmp_path / "lib.so.*gfx950")):
        text = subprocess.run([llvm, "-d", obj], check=True, stdout=subprocess.PIPE, text=True).stdout
        for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
            head = re.match(r"([0-9a-f]+) <(\S*fwd_splitkv_kernel\S*)>:", part)
            if not head:
                continue
            code = []
            for line in part.splitlines()[1:]:
                ins = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]{12}):", line)
                if ins:
                    jump = BRANCH.search(line)
                    code.append((int(ins[2], 16) - int(head[1], 16), ins[1], int(jump[1], 16) if jump else None))
            yield head[2], code


def _reaches_barrier(code):
    """Can the workgroup's next barrier be reached from the slot load without a wait for all of a wave's loads?"""
    at = {off: i for i, (off, _, _) in enumerate(code)}
    todo = [i + 1 for i, (_, ins, _) in enumerate(code) if ins.startswith(SLOT_LOAD)]
    assert todo, "no slot load"
    seen = set()
    while todo:
        i = todo.pop()
        if i in seen:
            continue
        seen.add(i)
        _, ins, target = code[i]
        if ins.startswith("s_barrier"):
            return True
        if (ins.startswith("s_waitcnt") and "vmcnt(0)" in ins) or ins.startswith("s_endpgm"):
            continue
        if ins.startswith(("s_branch", "s_cbranch")):
            todo.append(at[target])
        if not ins.startswith("s_branch"):
            todo.append(i + 1)
    return False


def test_every_path_to_the_barrier_waits_for_the_slot_words(tmp_path):
    """The wave that fetches the words may have neither a packed unit nor a window tile of its own (a split without work), and
    then nothing in between waits for memory unless the source says so; a barrier alone waits for LDS only."""
    kernels = dict(_kernels(tmp_path))
    assert len(kernels) == 108
    assert [name for name, code in kernels.items() if _reaches_barrier(code)] == []
