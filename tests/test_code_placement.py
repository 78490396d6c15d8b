"""Where the main loops of two GEMM kernels lie in the built library, within the 32-byte windows in which
instructions are fetched: csrc/gemm_main.h (place_main_loop) has the times.  A change of that file or of
the compiler that moves a loop shows here, and its padding is then chosen again."""
import os
import re
import shutil
import subprocess

import pytest

from flydsl_amd import _lib
from flydsl_amd.build import OUT, hipcc

OBJDUMP = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc()))), "llvm", "bin", "llvm-objdump")
# template arguments BM, BN, WM, WN, kind (int8 1, int4 2), epilogue (row x column scales), out_bf16, K tiles per
# step -> bytes into a window at which the smallest loop with matrix instructions may start
PLACES = {"ILi256ELi256ELi2ELi4ELi1ELi0ELb%dELi1EE": (0, 4), "ILi64ELi128ELi1ELi4ELi2ELi0ELb%dELi1EE": (16, 20, 24)}


def _main_loop(lines):
    """Offset of the smallest loop that holds matrix instructions (a backward branch and its target)."""
    at = [int(m.group(1), 16) if (m := re.search(r"//\s*([0-9A-Fa-f]+):", x)) else None for x in lines]
    loops = []
    for i, x in enumerate(lines):
        m = re.search(r"branch.*<\S+\+0x([0-9a-f]+)>", x)
        if m and at[i] is not None:
            start = at[0] + int(m.group(1), 16)
            if start <= at[i] and any("v_mfma" in y for y, a in zip(lines, at) if a is not None and start <= a <= at[i]):
                loops.append((at[i] - start, start))
    return min(loops)[1]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler of the toolchain")
def test_main_loops_lie_where_they_were_measured_fastest(tmp_path):
    _lib.load()
    so = shutil.copy(OUT, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", so], check=True, capture_output=True, cwd=tmp_path)
    objs = [str(tmp_path / f) for f in sorted(os.listdir(tmp_path)) if "gfx950" in f]
    names = {f"_ZN7flygemm16gemm_main_kernel{t % bf16}EvNS_8GemmArgsE": at for t, at in PLACES.items() for bf16 in (0, 1)}
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names), *objs],
                          check=True, capture_output=True, text=True).stdout
    found = {}
    for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
        m = re.match(r"[0-9a-f]+ <(\S+)>:\n", part)
        if m and m.group(1) in names:
            found[m.group(1)] = _main_loop(part[m.end():].strip("\n").split("\n")) % 32
    assert found.keys() == names.keys()
    for name, at in names.items():
        assert found[name] in at, (name, found[name])
