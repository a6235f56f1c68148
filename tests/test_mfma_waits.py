"""The wait between a matrix instruction and the first vector instruction that takes its results, in the built library.

The key pass of the running-softmax backward writes its score products in inline assembly, for which the compiler counts no wait
states: one that reads them early works as long as something else holds it up, and no comparison of results shows it.
So the machine code of flash.hip's kernels itself is looked at: twelve wait states between a 32 x 32 x 16 MFMA and a vector or memory
instruction, or another MFMA's factors, on its results (an instruction counts as one, s_nop n as n + 1), which is what the compiler puts
behind the MFMAs that it knows.
"""
import os
import re
import shutil
import subprocess

import pytest

from rtp_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT = 12

_REG = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")


def _registers(text):
    out = set()
    for kind, one, lo, hi in _REG.findall(text):
        out.update((kind, r) for r in (range(int(lo), int(hi) + 1) if lo else (int(one),)))
    return out


def early_readers(listing):
    """(kernel, instruction, wait states) of every instruction that touches an MFMA's results too early."""
    found, kernel, pending = [], None, []  # pending: [registers, wait states since]
    for line in listing.splitlines():
        m = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if m:
            kernel, pending = m.group(1), []
            continue
        text = line.split("//")[0].strip()
        if not text or not line[0].isspace():
            continue
        name, _, operands = text.partition(" ")
        mfma = name.startswith("v_mfma")
        if mfma:  # its addend is handed on inside the matrix pipe
            parts = re.split(r",\s*(?![^\[]*\])", operands)
            touched = _registers(" ".join(parts[1:3]))
        else:
            touched = _registers(operands) if not name.startswith("s_") else set()
        found += [(kernel, text, age) for regs, age in pending if age < WAIT and regs & touched]
        states = int(operands, 0) + 1 if name == "s_nop" else 1
        pending = [(regs, age + states) for regs, age in pending if age + states < WAIT]
        if name.startswith("v_mfma_f32_32x32x16"):
            regs = _registers(parts[0])
            pending = [(r, age) for r, age in pending if not r & regs] + [(regs, 0)]
        if name in ("s_branch", "s_endpgm", "s_setpc_b64"):
            pending = []
    return found


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler for gfx950 here")
    where = tmp_path_factory.mktemp("code")
    shutil.copy(_lib.LIB_PATH, where / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=where, check=True, capture_output=True)
    for f in sorted(where.glob("lib.so.*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", f.name], cwd=where, check=True, capture_output=True, text=True).stdout
        if "flash_dkv_kernel" in text:
            return text
    raise AssertionError("no object with the running-softmax kernels in " + _lib.LIB_PATH)


def test_results_are_taken_behind_their_wait(listing):
    assert len(re.findall(r"^[0-9a-f]+ <\S*flash_dkv_kernel", listing, re.M)) >= 6
    assert listing.count("v_mfma_f32_32x32x16") > 1000
    assert early_readers(listing) == []


def test_an_early_reader_is_found():
    head = "0000000000000000 <kernel>:\n\tv_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], 0\n"
    reader = "\tv_fmac_f32_e32 v30, s25, v3\n"
    other = "\tv_mfma_f32_32x32x16_bf16 v[32:47], v[20:23], v[24:27], 0\n"
    assert [age for _, _, age in early_readers(head + other + reader + "\ts_nop 10\n")] == [1]
    assert [age for _, _, age in early_readers(head + "\ts_nop 10\n" + reader)] == [11]
    assert early_readers(head + "\ts_nop 11\n" + reader) == []
    assert early_readers(head + other + "\ts_nop 10\n" + reader) == []
    # the same sum continued is no reader; a factor is
    assert early_readers(head + "\tv_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], v[0:15]\n") == []
    assert len(early_readers(head + "\tv_mfma_f32_32x32x16_bf16 v[48:63], v[0:3], v[24:27], 0\n")) == 1
