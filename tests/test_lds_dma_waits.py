"""The wait states that LDS loads issued from inline assembly must bring with them (the
compiler inserts none there), read from the compiled kernels' assembly: at least one
instruction between a write of M0 and the LDS load, and five wait states between a vector
instruction's write of an SGPR and a memory instruction that takes it as its base."""

from __future__ import annotations

import os
import re
import subprocess

import pytest

from helion_amd import _build

SOURCES = ("attention.hip", "linear_ce.hip")
BASE = re.compile(r"^global_load_lds_\w+ v\d+, s\[(\d+):(\d+)\]")
DEST = re.compile(r"^\S+ s(?:(\d+)|\[(\d+):(\d+)\])(?:,|$)")


def _instructions(text):
    for line in text.splitlines():
        t = line.split(";")[0].strip()
        if t and not t.endswith(":") and not t.startswith((".", "#")):
            yield t


def _faults(text):
    """(number of LDS loads, the faulty ones with the instructions before them)."""
    past, n, bad = [], 0, []
    for t in _instructions(text):
        if t.startswith("global_load_lds_"):
            n += 1
            ok = re.match(r"^s_\S+ m0,", past[-1]) is None
            base = BASE.match(t)
            for reg in range(int(base[1]), int(base[2]) + 1) if base else ():
                waits = 0
                for p in reversed(past):
                    d = DEST.match(p)
                    if d and int(d[1] or d[2]) <= reg <= int(d[1] or d[3]):
                        ok &= p.startswith("s_") or waits >= 5  # the register's last writer
                        break
                    nop = re.match(r"^s_nop (\d+)", p)
                    waits += 1 + int(nop[1]) if nop else 1
                    if waits >= 5:
                        break
            if not ok:
                bad.append(past[-5:] + [t])
        past.append(t)
        del past[:-8]
    return n, bad


def test_the_check_sees_missing_waits():
    ok = "s_mov_b32 m0, s1\ns_mov_b64 s[2:3], s[4:5]\nglobal_load_lds_dwordx4 v1, s[2:3]"
    assert _faults(ok) == (1, [])
    assert _faults("v_readfirstlane_b32 s2, v0\n" + ok) == (1, [])
    no_m0 = "s_mov_b64 s[2:3], s[4:5]\ns_mov_b32 m0, s1\nglobal_load_lds_dwordx4 v[2:3], off"
    no_base = "v_readfirstlane_b32 s3, v0\ns_mov_b32 m0, s1\ns_nop 0\nglobal_load_lds_dwordx4 v1, s[2:3]"
    for text in (no_m0, no_base):
        assert len(_faults(text)[1]) == 1


@pytest.mark.parametrize("src", SOURCES)
def test_lds_loads_wait(src, tmp_path):
    out = tmp_path / "k.s"
    flags = [f for f in _build.COMPILE_FLAGS if f != "-Wall"]
    subprocess.run([_build.HIPCC, *flags, "--cuda-device-only", "-S",
                    os.path.join(_build.SRC_DIR, src), "-o", str(out)],
                   check=True, capture_output=True)
    n, bad = _faults(out.read_text())
    assert n > 100
    assert not bad, f"{len(bad)} of {n}, the first:\n" + "\n".join(bad[0])
