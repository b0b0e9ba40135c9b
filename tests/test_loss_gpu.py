"""The runtime's softmax and loss kernel (tokamak_amd/csrc/tkm_rt_kernels.hip) alone, against the same in
float64: gradients, losses and counts of correct rows, over its vector forms (rows of a multiple of 8
columns, up to 2048 and up to 8192) and its general one, with ties and infinities among the logits.

Bounds: an exponential carries the roundings of its argument (2^-24 of the distance to the maximum) and
its own few, the sum at most `cols` roundings, each gradient a few of the magnitudes it is formed from;
the stored gradient adds its unit roundoff, 2^-11 in fp16 (2^-25 below the normal range), 2^-8 in bf16."""
import ctypes

import pytest

from attn_cases import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", (0, 1))
@pytest.mark.parametrize("kind", (0, 1, 2))
@pytest.mark.parametrize("cols", (8, 77, 520, 2048, 2056, 8192))
def test_softmax_loss(gpu, cols, kind, bf16):
    import torch
    from tokamak_amd import runtime as R
    f = R.lib().tkm_rt_softmax_loss
    dt, rows, gamma = (torch.bfloat16 if bf16 else torch.float16), 133, 2.0
    log(f"[case] cols {cols} kind {kind} bf16={bf16}")
    torch.manual_seed(cols + kind)
    x = (3 * torch.randn(rows, cols, device="cuda")).to(dt)
    y = torch.randint(0, cols, (rows,), device="cuda").to(torch.int32)
    best = x.float().argmax(1).to(torch.int32)
    y[::3] = best[::3]                                   # the label holds the maximum
    x[::6, cols - 1] = x[::6].amax(1)                    # and the last column does too
    y[6::12] = cols - 1
    x[1::9, 0] = float("-inf")
    x[5] = 0.5                                           # all columns alike
    y[5] = 0
    dx = torch.full((rows + 2, cols), float("nan"), dtype=dt, device="cuda")
    row_loss = torch.empty(rows, device="cuda")
    row_ok = torch.empty(rows, dtype=torch.int32, device="cuda")
    out, ok = torch.zeros(1, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for is_eval in (0, 1):
        assert f(p(x), bf16, p(y), 1, ctypes.c_void_p(dx.data_ptr() + dx.stride(0) * 2), p(row_loss), p(row_ok), rows,
                 cols, is_eval, rows - 20, kind, ctypes.c_float(gamma), p(out), p(ok), 0, 0, st) == 0
        torch.cuda.synchronize()
        want = x.double().argmax(1)
        want = torch.where((x == x.amax(1, keepdim=True)).double().argmax(1) == y, 1, 0)
        if is_eval:
            want[rows - 20:] = 0
        assert torch.equal(row_ok, want.to(torch.int32))
        assert int(ok) == int(want.sum())
        if is_eval:
            continue
        assert torch.isnan(dx[0]).all() and torch.isnan(dx[-1]).all(), "wrote outside dlogits"
        d = x.double() - x.double().amax(1, keepdim=True)
        q = torch.softmax(x.double(), 1)
        t = torch.zeros_like(q).scatter_(1, y.long()[:, None], 1.0)
        tp = (q * t).sum(1, keepdim=True).clamp(min=1e-7)
        if kind == 2:
            brier = (q * (q - t)).sum(1, keepdim=True)
            g, mag = 2 / cols * q * (q - t - brier), 2 / cols * q * (q + t + (q * (q + t)).sum(1, keepdim=True))
            loss = ((q - t) ** 2).sum(1) / cols
        else:
            fs = 1.0 if kind == 0 else (1 - tp) ** gamma - gamma * tp * (1 - tp) ** (gamma - 1) * tp.log()
            fm = 1.0 if kind == 0 else 1 - gamma * tp * tp.log()
            g, mag = fs * (q - t), fm * (q + t)
            loss = (-tp.log() * ((1 - tp) ** gamma if kind else 1.0))[:, 0]
        u = 2.0 ** -24 * (16 + cols + d.abs().nan_to_num(posinf=0.0))
        bound = (4 * u * mag + (2.0 ** -8 if bf16 else 2.0 ** -11) * g.abs()) / rows + (0 if bf16 else 2.0 ** -25)
        err = (dx[1:-1].double() - g / rows).abs()
        bad = int((~(err <= bound + 2.0 ** -126)).sum())
        log(f"    dlogits: max err {float(err.max()):.3e}, {bad} past the bound")
        assert bad == 0
        lb = 2.0 ** -24 * (64 + 2 * cols) * (1 + d.abs().nan_to_num(posinf=0.0).amax(1)) * (1 + loss) / rows
        assert bool(((row_loss.double() - loss / rows).abs() <= lb).all())
        assert abs(float(out) - float(loss.sum() / rows)) <= float(lb.sum()) + 1e-6 * float(loss.sum() / rows)
