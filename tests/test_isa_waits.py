"""Counted waits of the compiled kernels: a wait for asynchronous copies that leaves N younger loads in flight needs N of them behind the last copy."""
import os
import re
import shutil
import subprocess

import pytest

from mortar_amd import build

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
LOAD = re.compile(r"\s(?:buffer|global|flat|scratch)_load_\w+")


def _kernels(text):
    """{symbol: lines of its body} of a device assembly file."""
    out = {}
    for m in re.finditer(r"^(_Z\S+):.*?^\.Lfunc_end", text, re.M | re.S):
        out[m.group(1)] = m.group(0).splitlines()
    return out


def check_counted_wait(lines):
    """The hand-written wait behind the copies of a kernel: (loads it leaves in flight, loads issued behind the last copy)."""
    inline, wait = False, None
    for i, line in enumerate(lines):
        if "#ASMSTART" in line or "#ASMEND" in line:
            inline = "#ASMSTART" in line
        m = re.search(r"s_waitcnt vmcnt\((\d+)\)", line)
        if inline and m:
            wait = i, int(m.group(1))
            break
    assert wait, "no hand-written wait"
    last = max(i for i in range(wait[0]) if "global_load_lds" in lines[i])
    between = lines[last + 1:wait[0]]
    assert not any(re.search(r"\bs_c?branch", line) for line in between), "the loads behind the copies are not on every path"
    return wait[1], sum(bool(LOAD.search(line)) for line in between)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_tile_has_landed_when_the_values_are_multiplied(tmp_path):
    asm = tmp_path / "values.s"
    subprocess.run([HIPCC, *build.FLAGS, "-x", "hip", "--cuda-device-only", "-S", os.path.join(build.CSRC, "mortar_values.hip"), "-o", str(asm)],
                   check=True, capture_output=True)
    text = asm.read_text()
    kernels = {k: v for k, v in _kernels(text).items() if "values_resident_kernel" in k}
    assert len(kernels) >= 4
    for name, lines in kernels.items():
        left, behind = check_counted_wait(lines)
        assert left == 10 and behind >= left, (name, left, behind)


def test_a_missing_load_is_noticed():
    head = ["\t;;#ASMSTART", "\tglobal_load_lds_dwordx4 v[0:1], off", "\t;;#ASMEND"]
    tail = ["\t;;#ASMSTART", "\ts_waitcnt vmcnt(2)", "\t;;#ASMEND"]
    load = ["\tbuffer_load_dwordx4 v[4:7], v0, s[0:3], 0 offen"]
    assert check_counted_wait(head + load + load + tail) == (2, 2)
    assert check_counted_wait(head + load + tail) == (2, 1)
