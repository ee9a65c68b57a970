"""Checks on the gfx950 assembly that hipcc makes of the kernels' sources
(hipcc cross-compiles, so they need no GPU): what the memory model asks for
and a run would show only now and then."""
import os
import re
import subprocess

import pytest

from starpu_amd import _build

HIP = os.path.join(_build.CSRC, "hip")


def sources_with_agent_release():
    out = []
    for f in sorted(os.listdir(HIP)):
        if f.endswith(".hip"):
            with open(os.path.join(HIP, f)) as h:
                if re.search(r"ATOMIC_RELEASE, (\"agent\"|__HIP_MEMORY_SCOPE_AGENT)", h.read()):
                    out.append(f)
    return out


@pytest.mark.parametrize("src", sources_with_agent_release())
def test_l2_write_back_is_waited_for_before_the_next_store(src, tmp_path):
    # an agent-scope release writes the L2 back (buffer_wbl2) and then raises
    # a flag: without a wait for the write-back between the two, another
    # XCD can see the flag and read memory that the data has not reached
    asm = str(tmp_path / "k.s")
    subprocess.run(["hipcc", *_build.HIPCC_FLAGS, "-w", f"-I{_build.INCLUDE}", "--cuda-device-only", "-S", "-o", asm,
                    os.path.join(HIP, src)], check=True, stderr=subprocess.DEVNULL)
    with open(asm) as h:
        code = [l.strip() for l in h if l.startswith("\t") and not l.startswith("\t.") and not l.startswith("\t;")]
    found, bad = 0, []
    for i, l in enumerate(code):
        if not l.startswith("buffer_wbl2"):
            continue
        found += 1
        for nxt in code[i + 1:]:
            if re.match(r"s_waitcnt\b.*vmcnt\(0\)", nxt):
                break
            if re.match(r"(global|flat|buffer|scratch)_(store|atomic)|s_(c?branch|setpc|endpgm)", nxt):
                bad.append(f"{l} -> {nxt}")
                break
    assert found > 0 and not bad, (found, bad)
