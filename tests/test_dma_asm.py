"""The HBM -> LDS requests that the HIP kernels issue from inline assembly (attn_common.h), in the code that
the compiler makes of each source: every block names m0 as written, and holds by itself the wait states
that the hardware asks for, since the compiler's hazard pass does not look into it.  The
block must have 5 wait states before its first request (a VALU lane read, as of a spilled descriptor word,
may stand right before it) and 1 between a write of m0 and the request that uses it.  The GEMM kernels
wait the 5 states in a block of their own, once per step and pair of descriptors, and so may not spill
scalars: nothing else writes a descriptor's words by the vector unit after it."""
import os
import re
import subprocess

import pytest

from tokamak_amd import build as tb

SOURCES = ("attn_fwd.hip", "attn_bwd.hip", "tkm_gemm_mfma.hip")


def device_code(src, *args):
    cmd = [tb.hipcc(), *tb.HIPFLAGS, "--cuda-device-only", "-S", os.path.join(tb.CSRC, src), "-o", "-", *args]
    return subprocess.run(cmd, capture_output=True, text=True, check=True)


def asm_statements(ir):
    """(template, constraints) of the distinct asm statements."""
    found = set(re.findall(r'asm sideeffect "((?:[^"\\]|\\.)*)", "([^"]*)"', ir))
    return [(t.replace("\\0A", "\n").replace("\\09", "\t"), c) for t, c in found]


def wait_states(line):
    m = re.match(r"s_nop (\d+)", line)
    return int(m.group(1)) + 1 if m else 1


@pytest.mark.parametrize("src", SOURCES)
def test_requests_wait_for_their_operands(src):
    ir = device_code(src, "-emit-llvm").stdout
    assert ir.count("ptr.buffer.load.lds") == 0, "requests outside the asm, whose m0 the compiler writes"
    statements = asm_statements(ir)
    got = [(t, c) for t, c in statements if "buffer_" in t]
    assert got, "no request found"
    late = []
    for text, constraints in got:
        assert "~{m0}" in constraints, f"m0 is written and not named: {text!r}"
        assert "s_add" not in text or "~{scc}" in constraints, f"scc is written and not named: {text!r}"
        since_start, since_m0, requests = 0, None, 0
        for line in (x.strip() for x in text.split("\n")):
            if line.startswith("buffer_"):
                assert line.endswith("lds") and since_m0 is not None and since_m0 >= 1, f"m0 used too early: {text!r}"
                if since_start < 5:
                    late.append(text)
                requests += 1
            since_start += wait_states(line)
            since_m0 = 0 if re.match(r"s_\w+ m0,", line) else (None if since_m0 is None else since_m0 + wait_states(line))
        assert requests
    if late:
        assert src == "tkm_gemm_mfma.hip", f"requests without the wait for their descriptor: {late!r}"
        assert ("s_nop 4", "s,s") in statements, "no wait for the descriptors"
        usage = device_code(src, "-Rpass-analysis=kernel-resource-usage").stderr
        spills = re.findall(r"SGPRs Spill: (\d+)", usage)
        assert spills and set(spills) == {"0"}, f"a spilled descriptor word would be read too early: {spills}"
