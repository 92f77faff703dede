"""Wait states around the load-to-LDS copies that are written in assembly, where the compiler's own
hazard handling does not reach: at least one between a scalar write of M0 and a load that reads it,
and at least five between a vector instruction's write of a scalar register and a load that uses it as
its base. Checked in the generated gfx950 code of every source that copies this way.
"""
import os
import re
import subprocess

import pytest

from fastcone_amd import build

SOURCES = ["fc_backproject.hip", "fc_katsevich.hip"]


def _scalars(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m[1])} if m else set()


def _operands(ins):
    parts = ins.split(None, 1)
    return [o.strip() for o in parts[1].split(",")] if len(parts) > 1 else []


def _wait_states(ins):
    m = re.fullmatch(r"s_nop (\d+)", ins)
    return int(m[1]) + 1 if m else 1


def hazards(asm):
    """Loads to LDS and those that come too early, in the order of the text (straight-line code)."""
    loads, early, before = 0, [], []
    for line in asm.splitlines():
        ins = line.split(";")[0].strip()
        if re.match(r"_Z\w+:", line):
            before = []
        if not ins or ins.startswith((".", "_Z")) or ins.endswith(":"):
            continue
        if "load_lds" in ins or ins.endswith(" lds"):
            loads += 1
            base = set().union(*map(_scalars, _operands(ins)))
            waited = 0
            for prev in reversed(before):
                dst = _operands(prev)[:1]
                if waited < 1 and prev.startswith("s_") and dst == ["m0"]:
                    early.append((prev, ins))
                if waited < 5 and prev.startswith("v_") and dst and _scalars(dst[0]) & base:
                    early.append((prev, ins))
                waited += _wait_states(prev)
                if waited >= 5:
                    break
        before = before[-8:] + [ins]
    return loads, early


def test_hazards_are_found():
    load = "\tglobal_load_lds_dword v0, s[4:5]\n"
    assert hazards("\ts_mov_b32 m0, s2\n\ts_nop 0\n" + load) == (1, [])
    assert len(hazards("\ts_mov_b32 m0, s2\n" + load)[1]) == 1
    assert len(hazards("\tv_readfirstlane_b32 s5, v1\n\ts_nop 3\n" + load)[1]) == 1
    assert hazards("\tv_readfirstlane_b32 s5, v1\n\ts_nop 4\n" + load) == (1, [])


@pytest.mark.parametrize("src", SOURCES)
def test_wait_states(src, tmp_path):
    out = tmp_path / "k.s"
    cmd = [build._hipcc()] + build.HIPCC_FLAGS + ["-w", "--cuda-device-only", "-S", "-x", "hip",
                                                  os.path.join(build.CSRC, src), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True)
    loads, early = hazards(out.read_text())
    assert loads > 0
    assert early == []
