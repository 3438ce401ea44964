"""Direct-to-LDS copies in the built device code: the copy reads its LDS address
from M0, and the hardware requires one wait state between a scalar write of M0
and such a load, and five between a vector instruction's write of a scalar
register and a load that takes it as its base. The compiler inserts them for the
loads it knows; those written as asm carry their own. Checked in the assembly of
the libraries built here (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

from nncpu_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LIBS = ["libnncpu_hip.so", "libnncpu_gemma.so", "libnncpu_calib.so"]


def wait_states(instruction):
    m = re.match(r"s_nop (\d+)", instruction)
    return int(m[1]) + 1 if m else 1


def faults(code):
    """(copies, those too close to a write of M0, those too close to a vector write of their base)."""
    copies, m0, base = 0, [], []
    before = []
    for line in code:
        if re.match(r"^[0-9a-f]+ <", line):
            name, before = line, []
            continue
        t = line.split("//")[0].strip()
        if not line.startswith("\t") or not t:
            continue
        if re.match(r"(global|buffer|scratch)_load_lds|buffer_load\S* .*\blds\b", t):
            copies += 1
            if before and re.match(r"\S+ m0\b", before[-1]):
                m0.append((name, before[-1], t))
            pair = re.search(r"s\[(\d+):(\d+)\]", t)
            left = {int(pair[1]), int(pair[2])} if pair else set()
            states = 0
            for p in reversed(before):
                if states >= 5 or not left:
                    break
                w = re.match(r"(\S+) s(\d+)\b", p) or re.match(r"(\S+) s\[(\d+):(\d+)\]", p)
                if w and not re.match(r"s_(cmp|bitcmp|store|set)", w[1]):  # a register written, not read
                    written = set(range(int(w[2]), int(w[len(w.groups())]) + 1))
                    if w[1].startswith("v_") and written & left:
                        base.append((name, p, t))
                        break
                    left -= written
                states += wait_states(p)
        before = (before + [t])[-8:]
    return copies, m0, base


def test_scan_sees_both_hazards():
    code = ["0000 <k>:", "\ts_mov_b32 m0, s1", "\tglobal_load_lds_dwordx4 v1, s[2:3]",
            "\ts_mov_b32 m0, s1", "\ts_nop 0", "\tglobal_load_lds_dwordx4 v1, s[2:3]",
            "\tv_readfirstlane_b32 s2, v0", "\ts_nop 3", "\tglobal_load_lds_dwordx4 v1, s[2:3]",
            "\tv_readfirstlane_b32 s2, v0", "\ts_nop 4", "\tglobal_load_lds_dwordx4 v1, s[2:3]",
            "\tv_readlane_b32 s2, v0, 0", "\ts_add_u32 s2, s2, s9", "\tglobal_load_lds_dwordx4 v1, s[2:3]"]
    copies, m0, base = faults(code)
    assert (copies, len(m0), len(base)) == (5, 1, 1)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_copies_keep_their_wait_states(tmp_path):
    total = 0
    for lib in LIBS:
        shutil.copy(os.path.join(os.path.dirname(_lib.LIB_PATH), lib), tmp_path)
        subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    for f in sorted(os.listdir(tmp_path)):
        if not f.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], cwd=tmp_path, check=True, capture_output=True,
                              text=True).stdout
        copies, m0, base = faults(text.splitlines())
        assert not m0 and not base, (f, len(m0), m0[:3], len(base), base[:3])
        total += copies
    assert total > 500
