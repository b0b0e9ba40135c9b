"""The split forms of the HIP attention kernels (attn_launch.h: pick_rows_form, pick_keys_form) at the edges
of the rule that picks them and of their tiles: grids just on either side of each bound, sequences that
leave groups of waves without a tile, one key tile, key lengths inside every group, GQA lists, and persistent
assembly launches of a little more than one round.  Bounds as the other attention tests'."""
import pytest

from attn_cases import log, run_gpu_case

pytestmark = pytest.mark.gpu

# B, S, Hq, Hkv, D, causal, kv_len
CASES = [
    (1, 65, 2, 1, 64, True, None), (1, 97, 3, 3, 64, False, None),            # two tiles of 64, four of 32
    (1, 129, 8, 2, 64, True, [67]), (2, 257, 4, 4, 64, False, [257, 31]),      # groups without a visible key
    (4, 513, 8, 2, 64, True, [513, 1, 300, 0]), (4, 505, 8, 8, 64, False, [505, 65, 33, 500]),
    (2, 1030, 8, 4, 64, True, None), (2, 1030, 4, 2, 64, False, [1030, 999]),
    (8, 300, 11, 11, 64, True, None), (8, 300, 10, 5, 64, False, None),        # q 264 and 240 of 256
    (1, 2100, 4, 1, 64, True, None),                                           # a long GQA list, 8x1
    (1, 770, 3, 1, 128, True, None), (1, 769, 6, 1, 128, False, [500]),        # D 128: 4x1 rows, 4x1 keys
    (2, 800, 8, 4, 128, True, [800, 33]), (4, 257, 16, 16, 128, False, None),  # 4x2; 2x4
    (8, 130, 9, 9, 128, True, None),
    (3, 600, 33, 3, 128, True, None),                                          # 297 items of 256 rows: 149 workgroups
]


@pytest.mark.parametrize("dtype", ("f16", "bf16"))
@pytest.mark.parametrize("case", CASES, ids=["B%d-S%d-%d-%d-D%d-c%d%s" % (c[:5] + (c[5], "-kv" if c[6] else ""))
                                              for c in CASES])
def test_forms(gpu, case, dtype):
    B, S, Hq, Hkv, D, causal, kv_len = case
    res = run_gpu_case(gpu, B, S, Hq, Hkv, D, dtype=dtype, causal=causal, kv_len=kv_len, mul=0.7, seed=S + Hq)
    bad = [(r["name"], r["n_bad"]) for r in res if r["n_bad"]]
    assert not bad, bad


# B, S, Hq, Hkv, causal; the kernels that the rules for 256 compute units give D 128 there: short grids on the
# split HIP forms, full ones and the smallest calls on the assembly, each stage by its own grid
PATHS = [((1, 770, 3, 1, True), "fwd_hip", "dq_hip", "dkdv_hip"), ((2, 800, 8, 4, True), "fwd_hip", "dq_hip", "dkdv_hip"),
         ((4, 257, 16, 16, False), "fwd_hip", "dq_hip", "dkdv_asm"), ((3, 600, 33, 3, True), "fwd_asm", "dq_asm", "dkdv_hip"),
         ((4, 512, 4, 2, True), "fwd_asm", "dq_hip", "dkdv_hip"), ((4, 1024, 16, 16, True), "fwd_asm", "dq_asm", "dkdv_asm")]


@pytest.mark.parametrize("dtype", ("f16", "bf16"))
@pytest.mark.parametrize("shape,fwd,dq,dkdv", PATHS, ids=["B%d-S%d-%d-%d-c%d" % p[0] for p in PATHS])
def test_d128_kernels_of_the_rule(gpu, shape, fwd, dq, dkdv, dtype):
    import torch
    from tokamak_amd import attn
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the shapes are at the rules' lines for 256 compute units")
    B, S, Hq, Hkv, causal = shape
    log(f"[case] kernels of B{B} S{S} Hq{Hq} Hkv{Hkv} D128 {dtype}")
    dt = torch.float16 if dtype == "f16" else torch.bfloat16
    qkv = torch.randn((B, S, (Hq + 2 * Hkv) * 128), device=gpu).to(dt)
    o, lse = attn.gqa_fwd(qkv, B, S, Hq, Hkv, 128, causal=causal)
    assert attn.last_kernels() == [fwd]
    attn.gqa_bwd(qkv, o, torch.randn_like(o), lse, B, S, Hq, Hkv, 128, causal=causal)
    assert attn.last_kernels() == [dq, dkdv]
    torch.cuda.synchronize()


@pytest.mark.parametrize("S,where", ((300, 280), (300, 5), (1100, 700)))
def test_nan_key_reaches_output_from_every_group(gpu, S, where):
    """A NaN in one key's V makes every row that sees the key NaN, whichever group of waves walks its
    tile; a NaN in K makes those rows' scores NaN.  Rows whose last tile ends before the key stay finite
    (within the key's tile of up to 64 a masked probability of zero still meets the NaN of V)."""
    import torch
    from tokamak_amd import attn
    log(f"[case] NaN at key {where} of {S}")
    for part in (1, 2):
        qkv = torch.randn((1, S, 3, 64), device=gpu).half()
        qkv[0, where, part] = float("nan")
        o, lse = attn.gqa_fwd(qkv.view(1, S, -1), 1, S, 1, 1, 64, causal=True)
        nan = torch.isnan(o[0]).all(dim=1)
        clean = where // 64 * 64
        assert bool(nan[where:].all()) and not bool(torch.isnan(o[0, :clean]).any())
        assert bool(torch.isfinite(lse[0, 0, :clean]).all())
