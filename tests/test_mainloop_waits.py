"""The K loops of the 16x16-block kernels wait for memory once a step, for the stage they read next.  A load that an epilogue may
leave on its way (into a register of the loop, on a path where nothing uses it) makes the compiler wait for all memory in
every step instead, at 1.1 to 1.45 times the time and the same bits; the library's own code shows it."""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

import torch_int._CUDA as C

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
TWO_STAGES = {(256, 192), (192, 256), (256, 256)}   # a step waits for all of the next one's copies
SPILLS = {(256, 288)}                               # waits for its registers as well


def _blocks(code):
    """The basic blocks of a kernel's disassembly, as lists of instructions."""
    lines = re.findall(r"^\t(\S[^/\n]*?)\s*// ([0-9A-F]+):([^\n]*)", code, flags=re.M)
    start = int(lines[0][1], 16)
    targets = {start + int(t, 16) for text, _, rest in lines if "branch" in text for t in re.findall(r"<\S+\+0x([0-9a-f]+)>", rest)}
    block = []
    for text, at, _ in lines:
        if int(at, 16) in targets and block:
            yield block
            block = []
        block.append(text)
        if "branch" in text:
            yield block
            block = []


def _loops(obj):
    """(rows, columns, epilogue, vmcnt waits) of every block of a gemm_pipe16q_kernel that copies and multiplies."""
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True, text=True).stdout
    out = []
    for code in re.split(r"^[0-9a-f]+ <", text, flags=re.M):
        cfg = re.match(r"_ZN2ti\d+gemm_pipe16q_kernel.*?Pipe16QCfgILi(\d+)ELi(\d+)ELi\dELi\dELi(\d)E", code)
        for block in _blocks(code) if cfg else ():
            if sum("v_mfma" in i for i in block) >= 10 and any("global_load_lds" in i for i in block):
                out.append((*map(int, cfg.groups()), re.findall(r"vmcnt\((\d+)\)", "\n".join(block))))
    return out


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_a_step_waits_for_memory_once(tmp_path):
    lib = shutil.copy(C.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True)
    with ThreadPoolExecutor(4) as pool:
        found = list(pool.map(_loops, sorted(tmp_path.glob("*gfx950*"))))
    loops = [loop for some in found for loop in some]
    odd = [(bm, bn, kind, waits) for bm, bn, kind, waits in loops if (bm, bn) not in SPILLS
           and (len(waits) > 1 or ("0" in waits and (bm, bn) not in TWO_STAGES))]
    assert len(loops) > 200 and odd == [], (len(loops), odd)
    assert not [loop for loop in loops if loop[:3] == (256, 256, 6)]   # batched products without a bias: 3 to 12 % slower there
