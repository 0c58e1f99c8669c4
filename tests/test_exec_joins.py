"""The built kernels, as listed by llvm-objdump: where lanes that a branch has turned off come on again.

A block that a skipped branch jumps to (s_cbranch_execz), or that a divergent loop falls out into (s_cbranch_execnz), turns
its lanes on with an s_or of exec. Spills and copies that the compiler puts ahead of that instruction are for all lanes
but reach only those that are still on, which are none or the branch's; the others then go on with what the register or
the scratch slot held before. (At the end of the shuffle of the fixed effects, when lane 0 alone ran it, the address of
the residual's words in the LDS was lost in this way.)"""
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import pytest

from bayesrrcmd_amd import _abi

OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")) if p and Path(p).exists()), None)
VECTOR = ("v_", "scratch_", "ds_", "global_", "buffer_", "flat_")
LANELESS = ("v_writelane", "v_readlane", "v_readfirstlane", "v_nop")
LEAVES = ("s_branch", "s_cbranch", "s_endpgm", "s_setpc", "s_barrier")


def early_work(listing):
    """(function, block, instructions) of the blocks with vector work ahead of the instruction that turns lanes on."""
    functions, code = {}, None
    for line in listing.splitlines():
        m = re.match(r"^[0-9a-f ]*<(.+)>:$", line)
        if m and re.match(r"^L\d+$", m.group(1)):
            code.append((m.group(1), None))
        elif m:
            code = functions.setdefault(m.group(1), [])
        else:
            ins = line.split("//")[0].strip()
            if code is not None and re.match(r"[a-z]", ins):
                code.append((None, ins))
    found = []
    for name, code in functions.items():
        joins = {ins.split()[1] for _, ins in code if ins and ins.startswith("s_cbranch_execz")}
        block, early = None, []
        for label, ins in code:
            if label:
                if label in joins:
                    block, early = label, []
                elif early or not block:
                    block = None
                continue
            op = ins.split()[0]
            if block:
                if re.match(r"s_or_b64 exec, exec,|s_or_saveexec", ins):
                    if early:
                        found.append((name, block, early))
                    block = None
                elif re.search(r"_saveexec|s_mov_b64 exec", ins) or op.startswith(LEAVES):
                    block = None
                elif op.startswith(VECTOR) and not op.startswith(LANELESS):
                    early.append(ins)
            if op == "s_cbranch_execnz":
                block, early = "after " + ins, []
    return found


def test_finds_early_work():
    listing = """
0000 <kernel>:
    s_and_saveexec_b64 s[0:1], vcc
    s_cbranch_execz L0
    v_mov_b32_e32 v1, 0
    {0}
0001 <L0>:
    s_or_b64 exec, exec, s[0:1]
    s_and_saveexec_b64 s[0:1], vcc
    s_cbranch_execz L1
0002 <L2>:
    v_add_u32_e32 v2, 1, v2
    s_cbranch_execnz L2
    {1}
    s_or_b64 exec, exec, s[2:3]
    v_mov_b32_e32 v3, v2
0003 <L1>:
    v_writelane_b32 v9, s0, 1
    {2}
    s_or_b64 exec, exec, s[0:1]
    s_endpgm
"""
    assert early_work(listing.format("s_nop 0", "s_mov_b32 s4, 0", "s_nop 0")) == []
    got = early_work(listing.format("s_nop 0", "v_mov_b32_e32 v5, v6", "scratch_store_dword off, v8, off offset:4"))
    assert [(b, e[0].split()[0]) for _, b, e in got] == [("after s_cbranch_execnz L2", "v_mov_b32_e32"),
                                                         ("L1", "scratch_store_dword")]


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
@pytest.mark.skipif(not _abi.LIB_PATH.exists(), reason="library not built")
def test_built_kernels(tmp_path):
    lib = tmp_path / "lib.so"
    shutil.copy(_abi.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", lib.name], cwd=tmp_path, check=True, capture_output=True)
    parts = sorted(tmp_path.glob("lib.so.*gfx950"))
    assert parts

    def listing(part):
        return subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--symbolize-operands", part], check=True,
                              capture_output=True, text=True).stdout

    found, kernels = [], 0
    with ThreadPoolExecutor(4) as pool:
        for text in pool.map(listing, parts):
            kernels += len(re.findall(r"^\w+ <_Z.*kernel.*>:$", text, re.M))
            found += early_work(text)
    assert kernels >= 50 and found == []
