"""CPU tier: in the built kernels, no instruction touches the destination of an
LDS read before the wait for it.

The kernels issue their LDS reads by hand (lds_dma.h), so the compiler takes a
read's destination as written at once: a copy of it that it places before the
s_waitcnt, to assemble an operand say, would move registers that the read has yet
to fill. The disassembly of the built library is read in order. The generated
64-row kernels are left out: alternative paths of theirs issue the same reads, and
their generator checks its own waits.
"""
import os
import re
import shutil
import subprocess

import pytest

import cuda_amd._lib as L

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _registers(operand):
    m = re.fullmatch(r"([av])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return frozenset()
    lo, hi = (m[2], m[2]) if m[2] else (m[3], m[4])
    return frozenset(f"{m[1]}{i}" for i in range(int(lo), int(hi) + 1))


def _early_uses(text):
    """(LDS reads seen, [(function, read, instruction)] of early uses)."""
    function, pending, reads, early = "", [], 0, []
    for line in text.splitlines():
        label = re.match(r"[0-9a-f]+ <(.+)>:", line)
        if label:
            if not re.match(r"L\d", label[1]):
                function, pending = label[1], []
            continue
        inst = line.split("//")[0].strip()
        op, _, rest = inst.partition(" ")
        if op in ("s_endpgm", "s_branch"):   # what follows is reached from elsewhere
            pending = []
        elif op == "s_waitcnt":
            n = re.search(r"lgkmcnt\((\d+)\)", inst)
            if n:   # LDS operations complete in order
                pending = pending[len(pending) - int(n[1]):] if int(n[1]) else []
        else:
            operands = [_registers(x) for x in re.split(r"[,\s]+", rest)]
            used = frozenset().union(*operands)
            early += [(function, read, inst) for dst, read in pending if dst & used]
            if op.startswith("ds_"):
                reads += op.startswith("ds_read")
                pending.append((operands[0] if op.startswith("ds_read") else frozenset(), inst))
    return reads, early


def test_an_early_copy_is_found():
    head = "0000 <kernel>:\n\tds_read_b64_tr_b16 v[4:5], v1\n\tds_read_b64 v[6:7], v2 offset:64 // 00: D8\n"
    use = "\tv_mfma_f32_16x16x32_bf16 v[8:11], v[4:7], v[12:15], v[8:11]\n"
    assert _early_uses(head + "\ts_waitcnt lgkmcnt(0)\n" + use) == (2, [])
    assert len(_early_uses(head + "\ts_waitcnt lgkmcnt(1)\n" + use)[1]) == 1
    assert len(_early_uses(head + "\tv_mov_b32_e32 v20, v5\n\ts_waitcnt lgkmcnt(0)\n" + use)[1]) == 1
    assert len(_early_uses(head + "\tv_mov_b32_e32 v6, 0\n\ts_waitcnt lgkmcnt(0)\n" + use)[1]) == 1


def test_built_kernels_wait_for_their_lds_reads(tmp_path):
    if not os.path.exists(L.LIB_PATH) or not os.path.exists(OBJDUMP):
        pytest.skip("library not built, or no llvm-objdump")
    shutil.copy(L.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(tmp_path / "lib.so")], check=True, capture_output=True)
    reads, early = 0, []
    for part in tmp_path.glob("lib.so.*gfx950"):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(part)], check=True, capture_output=True,
                              text=True).stdout
        n, found = _early_uses(text)
        reads += n
        early += [x for x in found if "prefill_w64" not in x[0]]
    assert reads > 5000
    assert not early, early[:5]
