"""The global -> LDS copies of the built library keep the two distances that
inline asm has to keep by itself: one instruction between the scalar write of
M0 and the copy that uses it, five wait states between a vector instruction's
write of the copy's scalar base and the copy."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from gllm_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
INSN = re.compile(r"^\t(\S+)\s*(.*?)\s*(?://.*)?$")


def _wait_states(op, args):
    return 1 + int(args, 0) if op == "s_nop" else 1


def _base_written(op, args, base):
    """A vector instruction that writes one of the scalar registers `base`."""
    if not op.startswith("v_"):
        return False
    m = re.match(r"s(?:(\d+)|\[(\d+):(\d+)\])", args)
    if not m:
        return False
    lo, hi = (int(m[1]),) * 2 if m[1] else (int(m[2]), int(m[3]))
    return lo <= base[1] and hi >= base[0]


def faults(lines):
    """(copies seen, offending instruction sequences) of a disassembly."""
    hist, seen, bad = [], 0, []
    for line in lines:
        m = INSN.match(line)
        if not m:
            hist = []                      # a label: nothing is known of what ran before
            continue
        op, args = m[1], m[2]
        if "load_lds" in op:
            seen += 1
            if hist and hist[-1][0].startswith("s_mov") and hist[-1][1].startswith("m0"):
                bad.append((hist[-1], (op, args)))
            b = re.search(r"s\[(\d+):(\d+)\]", args)
            if b:
                states = 0
                for o, a in reversed(hist):
                    if states >= 5:
                        break
                    if _base_written(o, a, (int(b[1]), int(b[2]))):
                        bad.append(((o, a), (op, args)))
                    states += _wait_states(o, a)
        hist = (hist + [(op, args)])[-8:]
    return seen, bad


def test_the_check_itself():
    mov, load = "\ts_mov_b32 m0, s4   // 00: ab", "\tglobal_load_lds_dwordx4 v1, s[6:7]"
    assert faults([mov, load]) == (1, [(("s_mov_b32", "m0, s4"), ("global_load_lds_dwordx4", "v1, s[6:7]"))])
    assert faults([mov, "\ts_nop 0", load]) == (1, [])
    lane = "\tv_readfirstlane_b32 s7, v3"
    assert len(faults([lane, mov, "\ts_nop 0", load])[1]) == 1
    assert faults([lane, "\ts_nop 2", mov, "\ts_nop 0", load]) == (1, [])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_built_library(tmp_path):
    so = tmp_path / "lib.so"
    shutil.copy(_lib.LIB_PATH, so)
    subprocess.run([OBJDUMP, "--offloading", str(so)], check=True, capture_output=True, cwd=tmp_path)
    seen = 0
    for obj in glob.glob(str(tmp_path / "lib.so.*gfx950")):
        p = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", obj], stdout=subprocess.PIPE, text=True)
        n, bad = faults(p.stdout)
        assert p.wait() == 0
        seen += n
        assert not bad, f"{len(bad)} of {n} in {os.path.basename(obj)}, the first {bad[0]}"
    assert seen > 0
