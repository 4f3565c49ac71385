"""The assembly of the built library.

The global -> LDS copies keep the two distances that inline asm has to keep by
itself: one instruction between the scalar write of M0 and the copy that uses
it, five wait states between a vector instruction's write of the copy's scalar
base and the copy.  And no kernel reads a vector or accumulation register that
nothing in it writes: the register allocator has lost a quarter of a matrix
operand that way in kernels short of registers, which gave NaN now and then.
"""
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


def _registers(text, kind):
    out = set()
    for one, lo, hi in re.findall(r"\b%s(?:(\d+)\b|\[(\d+):(\d+)\])" % kind, text):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return out


def never_written(lines):
    """{kernel: registers} that its instructions read and none of them writes."""
    found, name, ins = {}, None, []

    def close():
        for kind in "av":
            written, read = {0} if kind == "v" else set(), set()       # v0: the thread index
            for op, args in ins:
                ops = args.split(",")
                no_dst = ("load_lds" in op or op.startswith(("v_cmp", "v_readlane", "v_readfirstlane", "s_"))
                          or re.match(r"(scratch|global|ds|flat|buffer)_(store|write|atomic)", op))
                if not no_dst:
                    written |= _registers(ops[0], kind)
                    if "swap" in op:
                        written |= _registers(ops[1], kind)
                read |= _registers(args if no_dst else ",".join(ops[1:]), kind)
            if read - written:
                found.setdefault(name, []).extend(f"{kind}{r}" for r in sorted(read - written))

    for line in lines:
        m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if m:
            close()
            name, ins = m[1], []
        elif (m := INSN.match(line)):
            ins.append((m[1], m[2]))
    close()
    return found


def test_the_register_check_itself():
    good = ["00 <k>:", "\tv_mov_b32 v1, v0", "\tv_accvgpr_write_b32 a2, v1", "\tds_write_b32 v0, a2"]
    assert never_written(good) == {}
    assert never_written(good + ["\tv_mfma_f32_16x16x4_f32 v[4:7], v1, a[2:3], 0"]) == {"k": ["a3"]}


@pytest.fixture(scope="module")
def disassembly(tmp_path_factory):
    """[(object, lines)] of the library's GPU code."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(_lib.LIB_PATH, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(d / "lib.so")], check=True, capture_output=True, cwd=d)
    objs = sorted(glob.glob(str(d / "lib.so.*gfx950")))
    assert objs
    ps = [subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", o], stdout=open(o + ".s", "w")) for o in objs]
    assert [p.wait() for p in ps] == [0] * len(ps)
    return [(os.path.basename(o), open(o + ".s").read().splitlines()) for o in objs]


def test_copies_wait_for_m0(disassembly):
    seen = 0
    for obj, lines in disassembly:
        n, bad = faults(lines)
        seen += n
        assert not bad, f"{len(bad)} of {n} in {obj}, the first {bad[0]}"
    assert seen > 0


def test_every_register_read_is_written(disassembly):
    for obj, lines in disassembly:
        assert never_written(lines) == {}, obj
