"""The bands of rows that the generated backwards are cut into (tkm_bwd_band, tkm_bwd_bands): whole passes of
a block, all rows covered by bands of which none is empty, and no more of them than a workspace sized for
one band per 4 rows and 2048 blocks holds.  Host code, no GPU; the functions are hidden in the libraries, so
their source is compiled here with two names of its own."""
import ctypes
import os
import subprocess

import pytest

from tokamak_amd import build as tb


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("bands")
    src, so = os.path.join(d, "bands.c"), os.path.join(d, "bands.so")
    with open(src, "w") as f:
        f.write('#include "%s"\n' % os.path.join(tb.CSRC, "tkm_prep_codegen.c"))
        f.write("#define VISIBLE __attribute__((visibility(\"default\")))\n")
        f.write("VISIBLE int band(int r, int x, int s, int p) { return tkm_bwd_band(r, x, s, p); }\n")
        f.write("VISIBLE int bands(int r, int b) { return tkm_bwd_bands(r, b); }\n")
    rest = [os.path.join(tb.CSRC, s) for s in ("tkm_codegen_util.c", "tkm_error.c", "tkm_prelude.c")]
    subprocess.run(["gcc", *tb.CFLAGS, "-shared", src, *rest, "-o", so, "-lm"], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("partials", (0, 1))
@pytest.mark.parametrize("side", (4, 8, 16, 32, 64, 256))
def test_bands_are_whole_passes(rule, side, partials):
    # 100 rows of 32 a pass, 4096 of 80 blocks and 16384 of 24: an even share of them is not whole passes
    rows = list(range(0, 600)) + [1027, 2048, 4096, 4099, 16384, 199999, 1 << 24]
    for x in (1, 2, 3, 5, 9, 24, 80, 257):
        for r in rows:
            band = rule.band(r, x, side, partials)
            bands = rule.bands(r, band)
            assert band >= side and band % side == 0, (r, x, band)
            assert bands >= 1 and bands * band >= r and (bands == 1 or (bands - 1) * band < r), (r, x, band, bands)
            assert bands <= max(1, min((r + 3) // 4, -(-(2048 if partials else 16384) // x))), (r, x, bands)
