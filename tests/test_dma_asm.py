"""The HBM -> LDS requests that the HIP kernels issue from inline assembly (attn_common.h), in the code that
the compiler makes of each source: every block names m0 as written, and holds by itself the wait states
that the hardware asks for, since the compiler's hazard pass does not look into it.  Of its own accord the
block must have 5 wait states before its first request (a VALU lane read, as of a spilled descriptor word,
may stand right before it) and 1 between a write of m0 and the request that uses it."""
import os
import re
import subprocess

import pytest

from tokamak_amd import build as tb

SOURCES = ("attn_fwd.hip", "attn_bwd.hip", "tkm_gemm_mfma.hip")


def blocks(src):
    """(template, constraints) of the distinct asm statements with a buffer request in a source's device code."""
    cmd = [tb.hipcc(), *tb.HIPFLAGS, "--cuda-device-only", "-emit-llvm", "-S", os.path.join(tb.CSRC, src), "-o", "-"]
    ir = subprocess.run(cmd, capture_output=True, text=True, check=True).stdout
    found = set(re.findall(r'asm sideeffect "((?:[^"\\]|\\.)*)", "([^"]*)"', ir))
    assert ir.count("ptr.buffer.load.lds") == 0, "requests outside the asm, whose m0 the compiler writes"
    return [(t.replace("\\0A", "\n").replace("\\09", "\t"), c) for t, c in found if "buffer_" in t]


def wait_states(line):
    m = re.match(r"s_nop (\d+)", line)
    return int(m.group(1)) + 1 if m else 1


@pytest.mark.parametrize("src", SOURCES)
def test_requests_wait_for_their_operands(src):
    got = blocks(src)
    assert got, "no request found"
    for text, constraints in got:
        assert "~{m0}" in constraints, f"m0 is written and not named: {text!r}"
        since_start, since_m0, requests = 0, None, 0
        for line in (x.strip() for x in text.split("\n")):
            if line.startswith("buffer_"):
                assert line.endswith("lds") and since_start >= 5, f"{since_start} wait states at the start: {text!r}"
                assert since_m0 is not None and since_m0 >= 1, f"m0 used too early: {text!r}"
                requests += 1
            since_start += wait_states(line)
            since_m0 = 0 if re.match(r"s_\w+ m0,", line) else (None if since_m0 is None else since_m0 + wait_states(line))
        assert requests
        # an arithmetic step of m0 writes the carry
        assert "s_add" not in text or "~{scc}" in constraints, f"scc is written and not named: {text!r}"
