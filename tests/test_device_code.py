"""Wait states that the compiler does not insert: inside inline asm its hazard
handling ends, so what a statement needs has to stand in the statement."""
import os
import re
import subprocess

from ktir_cpu_amd import build


def _statements(src, tmp_path):
    """The instruction lists of the inline asm statements of csrc/`src`, as compiled for gfx950."""
    out = tmp_path / "device.txt"
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "-S", "--cuda-device-only", os.path.join(build.CSRC, src), "-o",
                    str(out)], check=True, capture_output=True)
    found = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", out.read_text(), re.S)
    return [[x.split(";")[0].strip() for x in f.splitlines() if x.split(";")[0].strip()] for f in found]


def test_loads_to_lds_wait_for_their_descriptor(tmp_path):
    """A vector instruction right before the statement may have written the
    descriptor's scalar registers: a load may read them five wait states later,
    and M0 one after it was written.  M0 is afterwards what it was."""
    stmts = [s for s in _statements("ktir_pattn_split.hip", tmp_path) if any(" lds" in x for x in s)]
    assert len(stmts) > 16
    for s in stmts:
        waits, m0_waits = 0, 0
        for x in s:
            op, _, rest = x.partition(" ")
            if op.startswith("buffer_load") and rest.endswith("lds"):
                assert waits >= 5 and m0_waits >= 1, s
            n = int(rest) + 1 if op == "s_nop" else 1
            waits, m0_waits = waits + n, m0_waits + n
            if rest.startswith("m0"):
                m0_waits = 0
        assert s[0].endswith(", m0") and s[-2] == f"s_mov_b32 m0, {s[0].split()[1].rstrip(',')}" and s[-1] == "s_nop 0", s
