"""The work this framework is used for, as timed and compared cases.

Each case is one pass through the public Python entry points: the attention calls of
``tokamak_amd.attn``, the generated epilogues of ``tokamak_amd.prep`` / ``tokamak_amd.plasma``,
and whole models through ``tokamak_amd.runtime.Runtime`` (a training step, an inference batch).
``listed()`` holds the sizes of the repository's own configurations and tests with ragged and
long relatives of them; ``draw`` gives more of the same ranges.

Kinds and their fields:
  attn   B, S, Hq, Hkv, D, dtype, causal, padded (per-batch key lengths), bwd (0: forward only),
         mul (scale of Q, K and V)
  layer  B, S, Hq, Hkv, D, C, F, dtype, qknorm, rope: the three epilogues of one decoder layer
         (qkv-prep; residual Add -> RMSNorm over C; SiLU(gate) * up over 2F), forward and backward
  step   model, B, S, dtype, host (1: rows and labels come from host memory each step)
  infer  model, B, S, dtype: host rows in, host logits out
"""
from __future__ import annotations

import json
import math
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DT = {"f16": torch.float16, "bf16": torch.bfloat16}
LR = 1e-2
MOMENTUM, DECAY = 0.9, 1e-4            # the runtime's SGD; the decay is on GEMM weights only

# Decoders of tests/golden/models, as the graphs of tests/golden/tkm_graphs.npz hold them:
# the largest batch and the sequence lengths a drawn case may take.
MODELS = {"cfg4": (8, 512), "induction": (8, 512), "llama_small": (16, 256)}


def listed():
    attn = {"kind": "attn", "padded": 0, "bwd": 1, "mul": 1.0, "causal": 1}
    return [
        # the smallest calls: the reference's CPU-checked shape, bound by launches and latency
        {**attn, "name": "attn-small", "B": 2, "S": 128, "Hq": 4, "Hkv": 4, "D": 64, "dtype": "f16"},
        # forward only (inference prefill) at head dim 64
        {**attn, "name": "attn-d64-fwd", "B": 4, "S": 1024, "Hq": 8, "Hkv": 8, "D": 64, "dtype": "f16",
         "bwd": 0, "mul": 0.5},
        # the attention layer of the 8-layer bf16 decoder below
        {**attn, "name": "attn-d64-layer-bf16", "B": 8, "S": 512, "Hq": 8, "Hkv": 8, "D": 64, "dtype": "bf16"},
        # long context at head dim 64, grouped heads
        {**attn, "name": "attn-d64-long-gqa", "B": 2, "S": 4096, "Hq": 16, "Hkv": 4, "D": 64, "dtype": "f16"},
        # a short batch at head dim 128: too few 256-row blocks to fill the chip
        {**attn, "name": "attn-d128-short", "B": 4, "S": 512, "Hq": 4, "Hkv": 2, "D": 128, "dtype": "f16"},
        # the headline shape: fp16 training at head dim 128
        {**attn, "name": "attn-d128", "B": 4, "S": 2048, "Hq": 16, "Hkv": 16, "D": 128, "dtype": "f16"},
        # ragged bf16 batch with grouped heads and padding
        {**attn, "name": "attn-d128-ragged-bf16", "B": 3, "S": 1531, "Hq": 16, "Hkv": 4, "D": 128,
         "dtype": "bf16", "padded": 1},
        # long documents, bidirectional, padded
        {**attn, "name": "attn-d128-long-padded", "B": 2, "S": 8192, "Hq": 32, "Hkv": 32, "D": 128,
         "dtype": "f16", "causal": 0, "padded": 1},
        # the generated epilogues of one decoder layer, training
        {"name": "layer-epilogues", "kind": "layer", "B": 8, "S": 512, "Hq": 8, "Hkv": 8, "D": 64, "C": 512,
         "F": 1376, "dtype": "bf16", "qknorm": 1, "rope": 1},
        # the whole training step of the 8-layer decoder, on data resident on the device
        {"name": "train-step", "kind": "step", "model": "cfg4", "B": 8, "S": 512, "dtype": "bf16", "host": 0},
        # the training step of a small model fed from the host: many short launches
        {"name": "train-step-small", "kind": "step", "model": "induction", "B": 4, "S": 512, "dtype": "f16",
         "host": 1},
        # inference of a small model, host rows in and logits out
        {"name": "infer-small", "kind": "infer", "model": "induction", "B": 4, "S": 512, "dtype": "f16"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(("attn", "layer", "step", "infer"), (60, 16, 12, 12))[0]
    if kind == "attn":
        most = work(listed()[7])["flops"]
        while True:
            hkv, g = rng.choice((1, 2, 4, 8, 16)), rng.choice((1, 1, 2, 4))
            c = {"kind": "attn", "B": _log_int(rng, 1, 8), "S": _log_int(rng, 64, 8192), "Hq": hkv * g, "Hkv": hkv,
                 "D": rng.choice((64, 128)), "dtype": rng.choice(("f16", "bf16")), "causal": int(rng.random() < 0.7),
                 "padded": int(rng.random() < 0.3), "bwd": int(rng.random() < 0.7), "mul": 1.0}
            if c["Hq"] <= 32 and c["B"] * c["S"] * c["Hq"] <= 524288 and work(c)["flops"] <= most:
                return c
    if kind == "layer":
        hkv, g, d = rng.choice((1, 2, 4, 8)), rng.choice((1, 2, 4)), rng.choice((64, 128))
        return {"kind": "layer", "B": _log_int(rng, 1, 8), "S": _log_int(rng, 32, 2048), "Hq": hkv * g, "Hkv": hkv,
                "D": d, "C": 64 * rng.randint(1, 32), "F": 32 * rng.randint(2, 160),
                "dtype": rng.choice(("f16", "bf16")), "qknorm": int(d == 64 and rng.random() < 0.5),
                "rope": int(rng.random() < 0.8)}
    model = rng.choice(("cfg4", "induction", "llama_small"))
    b, s = MODELS[model]
    c = {"kind": kind, "model": model, "B": _log_int(rng, 1, b), "S": _log_int(rng, 16, s),
         "dtype": rng.choice(("f16", "bf16"))}
    if kind == "step":
        c["host"] = rng.randint(0, 1)
        if model == "cfg4":              # fp16 holds no gradient of 8192 logits over as many rows
            c["dtype"] = "bf16"
    return c


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed, salt, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed) * 64 + salt)
    return g


def _randn(shape, seed, salt, mul=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=_gen(seed, salt), device="cuda") * mul).to(dtype)


def _kv_len(case, seed):
    """One full row and others of between half and all of the keys, as a padded batch has."""
    if not case["padded"]:
        return None
    n = torch.randint((case["S"] + 1) // 2, case["S"] + 1, (case["B"],), generator=_gen(seed, 9), device="cuda")
    n[0] = case["S"]
    return n.to(torch.int32)


def _attn_inputs(case, seed):
    dt = DT[case["dtype"]]
    w = (case["Hq"] + 2 * case["Hkv"]) * case["D"]
    qkv = _randn((case["B"], case["S"], w), seed, 1, case["mul"], dt)
    dout = _randn((case["B"], case["S"], case["Hq"] * case["D"]), seed, 2, 1.0, dt)
    return qkv, dout, _kv_len(case, seed)


def _layer_inputs(case, seed):
    dt, rows = DT[case["dtype"]], case["B"] * case["S"]
    nh = case["Hq"] + 2 * case["Hkv"]
    c, qk = nh * case["D"], (case["Hq"] + case["Hkv"]) * case["D"]
    t = {"x": _randn((rows, c), seed, 1, 1.0, dt), "dx": _randn((rows, c), seed, 2, 1.0, dt),
         "bias": _randn(c, seed, 3, 0.1), "gamma": 1 + _randn(qk, seed, 4, 0.1)}
    t["h"], t["res"] = _randn((rows, case["C"]), seed, 5, 1.0, dt), _randn((rows, case["C"]), seed, 6, 1.0, dt)
    t["dh"], t["w"] = _randn((rows, case["C"]), seed, 7, 1.0, dt), 1 + _randn(case["C"], seed, 8, 0.1)
    t["gu"], t["df"] = _randn((rows, 2 * case["F"]), seed, 10, 1.0, dt), _randn((rows, case["F"]), seed, 11, 1.0, dt)
    return t


# ---- models ---------------------------------------------------------------------------------

OP_TWIN, OP_QKV, OP_GQA, OP_RMSNORM, OP_PREP, OP_BIAS, OP_ADD, OP_MUL, OP_CE = 4, 5, 6, 29, 31, 32, 56, 57, 59
GEMM = (3, OP_TWIN, OP_QKV)
SIZEOF_NODE, GROUPS_AT, SIZEOF_GROUP, BATCH_AT, ARENA_AT = 264, 270340, 4296, 1370120, 1370128
_graphs = {}


def _graph(case):
    """(graph bytes, nodes) of the model at the case's batch and sequence length: the planner gives
    every stored node a slot of its own, so another size is the same plan with other slots."""
    if not _graphs:
        fx = np.load(os.path.join(ROOT, "tests", "golden", "tkm_graphs.npz"))
        for m in MODELS:
            _graphs[m] = (fx[m + "/graph"].tobytes(), bytes(fx[m + "/json"]).decode())
    raw, text = _graphs[case["model"]]
    raw, js = bytearray(raw), json.loads(text)

    def put(at, v, t=np.int32):
        raw[at:at + np.dtype(t).itemsize] = np.array([v], t).tobytes()

    off = 0
    for n in js["nodes"]:
        at = SIZEOF_NODE * n["id"]
        n["H"], n["W"] = 1, case["S"]
        put(at + 232, 1)
        put(at + 236, case["S"])
        if n["out_buf_id"] >= 0 and n["out_bytes"] > 0:
            size = 2 * case["B"] * case["S"] * n["C"]
            put(at + 248, off, np.uint64)
            put(at + 256, size, np.uint64)
            off += (size + 255) // 256 * 256
    for k in range(js["num_groups"]):
        put(GROUPS_AT + SIZEOF_GROUP * k + 100, 1)
        put(GROUPS_AT + SIZEOF_GROUP * k + 104, case["S"])
    put(BATCH_AT, case["B"])
    put(ARENA_AT, off, np.uint64)
    put(ARENA_AT + 8, off, np.uint64)
    nodes = js["nodes"]
    for n in nodes:
        n["C"] = n["C"] or (nodes[n["in0"]]["c_out"] or nodes[n["in0"]]["C"] if n["in0"] >= 0 else 0)
    if case["kind"] == "infer":          # the flow without its loss: it ends in the logits
        for n in nodes:
            if n["op"] == OP_CE:
                n["dead"] = 1
                put(SIZEOF_NODE * n["id"] + 48, 1)
    return bytes(raw), nodes


def _params(nodes):
    """[(node, kind, shape)] in the order of the model's weight file."""
    got = []
    for n in nodes:
        if n["op"] in GEMM:
            got.append((n, "W", (nodes[n["in0"]]["C"], n["C"])))
        if n["op"] in (OP_BIAS, OP_PREP):
            got.append((n, "bias", (n["C"],)))
        if n["op"] in (OP_RMSNORM, OP_PREP):
            got.append((n, "w", (n["C"],)))
    return got


def _weights(case, nodes, seed):
    """Weights as a training run starts with them: GEMM weights of the usual spread 0.02 (values of the
    16-bit type, as the step computes with them), small biases, norm weights around one."""
    g, got = _gen(seed, 20), []
    for _, kind, shape in _params(nodes):
        r = torch.randn(shape, generator=g, device="cuda")
        got.append((0.02 * r).to(DT[case["dtype"]]).float() if kind == "W" else
                   0.02 * r if kind == "bias" else 1 + 0.1 * r)
    return got


def _model_inputs(case, nodes, seed):
    rows, vocab = case["B"] * case["S"], [n for n in nodes if n["op"] in GEMM][-1]["C"]
    x = _randn((rows, nodes[0]["C"]), seed, 21, 1.0, DT[case["dtype"]]).float()
    y = torch.randint(0, vocab, (rows,), generator=_gen(seed, 22), device="cuda").to(torch.int32)
    return x, y


class _Device:
    """An fp32 device buffer of a runtime's, for torch.as_tensor; the runtime lives as long as its views."""

    def __init__(self, rt, ptr, shape):
        self.rt = rt
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False),
                                         "version": 2}


def _returned(nodes):
    """Indices into _params of the updated tensors a step returns: every live GEMM weight, then the live
    vectors in file order, as many as fit."""
    ps = _params(nodes)
    live = [k for k, (n, kind, _) in enumerate(ps) if not n["dead"] and not (n["op"] == OP_PREP and kind == "w")]
    mats = [k for k in live if ps[k][1] == "W"]
    return (mats + [k for k in live if ps[k][1] != "W"])[:62]


# ---- the passes -----------------------------------------------------------------------------


def prepare(case, seed):
    s = {"case": case}
    if case["kind"] == "attn":
        from tokamak_amd import attn
        attn.lib()
        s["qkv"], s["dout"], s["kv_len"] = _attn_inputs(case, seed)
        return s
    if case["kind"] == "layer":
        from tokamak_amd import plasma, prep
        t = s["t"] = _layer_inputs(case, seed)
        rows, dt, dev = case["B"] * case["S"], DT[case["dtype"]], t["x"].device
        s["prep"] = prep.Prep(case["Hq"], case["Hkv"], case["D"], case["S"], qknorm=bool(case["qknorm"]),
                              rope=bool(case["rope"]), dtype=case["dtype"], theta=10000.0)
        s["norm"] = plasma.Plasma(case["C"], ["Add", ("RMSNorm", 1e-5)], dtype=case["dtype"], group_id=1)
        s["ffn"] = plasma.Plasma(case["F"], (), True, ["SiLU"], (), dtype=case["dtype"], group_id=2)
        like = lambda k: torch.empty_like(t[k])  # noqa: E731
        s["tn"] = {"in": t["h"], ("branch", 0): t["res"], "out": like("h"), "dout": t["dh"], "din": like("h"),
                   ("dbranch", 0): like("h"), ("w", 1): t["w"], ("dw", 1): like("w"), ("xhat", 1): like("h"),
                   ("istd", 1): torch.empty((rows, (case["C"] + 63) // 64), dtype=torch.float32, device=dev)}
        s["tf"] = {"in": t["gu"], "out": like("df"), "dout": t["df"], "din": like("gu")}
        return s
    from tokamak_amd import runtime as R
    raw, nodes = _graph(case)
    dt = {"f16": 0, "bf16": 1}[case["dtype"]]
    rt = s["rt"] = R.Runtime(R.graph_buffer(raw), dtype=dt, training=case["kind"] == "step", token_labels=True)
    ws = _weights(case, nodes, seed)
    if not rt.load_weights(R.encode_weights([w.cpu().numpy() for w in ws])):
        raise RuntimeError("the weights do not fit the model")
    x, y = _model_inputs(case, nodes, seed)
    s["x"], s["y"] = x.cpu().numpy(), y.cpu().numpy()
    if case["kind"] == "step":
        if not case["host"]:
            rt.upload(s["x"], s["y"])
        import ctypes
        s["out"], ps = {}, _params(nodes)
        for k in _returned(nodes):
            master = ctypes.c_void_p()
            if R.lib().tkm_runtime_tensor(rt.rt, k, ctypes.byref(master), None, None, None, None):
                raise RuntimeError("the model has no tensor %d" % k)
            s["out"]["p%d" % k] = torch.as_tensor(_Device(rt, master.value, ps[k][2]), device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "attn":
        from tokamak_amd import attn
        shape = (case["B"], case["S"], case["Hq"], case["Hkv"], case["D"])
        o, lse = attn.gqa_fwd(s["qkv"], *shape, causal=bool(case["causal"]), kv_len=s["kv_len"])
        if not case["bwd"]:
            return {"o": o, "lse": lse}
        dqkv = attn.gqa_bwd(s["qkv"], o, s["dout"], lse, *shape, causal=bool(case["causal"]), kv_len=s["kv_len"])
        return {"o": o, "lse": lse, "dqkv": dqkv}
    if case["kind"] == "layer":
        t, rows = s["t"], case["B"] * case["S"]
        gamma = t["gamma"] if case["qknorm"] else None
        qkv, xhat, istd = s["prep"].fwd(t["x"], t["bias"], gamma)
        s["norm"].fwd(s["tn"], rows)
        s["ffn"].fwd(s["tf"], rows)
        s["ffn"].bwd(s["tf"], rows, 0)
        s["norm"].bwd(s["tn"], rows, 0)
        din, dgamma, dbias = s["prep"].bwd(t["dx"], xhat, istd, gamma)
        n, f = s["tn"], s["tf"]
        return {"qkv": qkv, "xhat": xhat, "istd": istd, "din": din, "dgamma": dgamma, "dbias": dbias,
                "norm": n["out"], "dh": n["din"], "dres": n[("dbranch", 0)], "dw": n[("dw", 1)],
                "ffn": f["out"], "dgu": f["din"]}
    if case["kind"] == "infer":
        return {"logits": s["rt"].forward(s["x"])}
    if case["host"]:
        return {"loss": s["rt"].step(s["x"], s["y"], LR), **s["out"]}
    s["rt"].step_device(LR)
    return s["out"]


# ---- what a pass cannot do without ------------------------------------------------------------


def work(case):
    e = 2
    if case["kind"] == "attn":
        B, S, Hq, Hkv, D = (case[k] for k in ("B", "S", "Hq", "Hkv", "D"))
        keys = S * (1 + (B - 1) * 0.75) / B if case["padded"] else S      # what _kv_len gives on average
        f = 4.0 * B * Hq * S * keys * D * (0.5 if case["causal"] else 1.0)
        qkv, o, lse = B * S * (Hq + 2 * Hkv) * D * e, B * S * Hq * D * e, B * S * Hq * 4
        if not case["bwd"]:
            return {"bytes": qkv + o + lse, "flops": f}
        return {"bytes": (qkv + o + lse) + (qkv + 2 * o + lse + qkv), "flops": 3.5 * f}
    rows = case["B"] * case["S"]
    if case["kind"] == "layer":
        c = (case["Hq"] + 2 * case["Hkv"]) * case["D"]
        nh = case["Hq"] + case["Hkv"]
        save = (nh * case["D"] * e + nh * 4) if case["qknorm"] else 0
        per = 4 * c * e + 2 * save                                          # x -> qkv, dqkv -> dx
        per += (3 + 4) * case["C"] * e + 2 * case["C"] * e + 2 * 4 * (case["C"] // 64)   # Add, RMSNorm, xhat
        per += 3 * case["F"] * e + 5 * case["F"] * e                        # gate, up -> ffn; gate, up, d -> d, d
        return {"bytes": float(rows * per), "flops": 0.0}
    _, nodes = _graph(case)
    flops = bytes_ = 0.0
    for n in nodes:
        if n["dead"]:
            continue
        if n["op"] in GEMM:
            K = nodes[n["in0"]]["C"]
            flops += 2.0 * rows * K * n["C"] * (3 if case["kind"] == "step" else 1)
            bytes_ += K * n["C"] * (22 + 2 * e if case["kind"] == "step" else e)
        if n["op"] == OP_GQA:
            f = 2.0 * case["B"] * n["q_heads"] * case["S"] ** 2 * n["head_dim"]
            flops += f * (3.5 if case["kind"] == "step" else 1)
        if n["out_buf_id"] >= 0 and n["out_bytes"] > 0:
            # a stored tensor is written and read once, in training its gradient too
            bytes_ += 2.0 * rows * n["C"] * e * (3 if case["kind"] == "step" else 1)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # About four times the difference measured between correct results at these precisions: storage
    # rounding of O, dQ, dK, dV and of 16-bit P and dS; in whole models, GEMM sums off by a few
    # fp32 roundings, which flip the 16-bit roundings of all that follows.
    bf = case["dtype"] == "bf16"
    if case["kind"] in ("attn", "layer"):
        return {"rel": 8e-3 if bf else 1.5e-3, "max": 0.2 if bf else 0.05}
    if case["kind"] == "infer":
        return {"rel": 0.03, "max": 0.5} if bf else {"rel": 4e-3, "max": 0.06}
    # the step's change of the weights, which grows as fewer rows average the gradient
    return {"rel": (3e-4 if bf else 3e-5) * max(1.0, math.sqrt(2048 / (case["B"] * case["S"])))}


# ---- the same in 64 bits ----------------------------------------------------------------------


def _heads(x, H, D):
    return x.reshape(x.shape[0], H, D)


def _exact_attn(case, seed):
    B, S, Hq, Hkv, D = (case[k] for k in ("B", "S", "Hq", "Hkv", "D"))
    qkv, dout, kv_len = _attn_inputs(case, seed)
    scale, g = float(np.float32(1.0) / np.sqrt(np.float32(D))), Hq // Hkv
    o = torch.zeros((B, S, Hq, D), dtype=torch.float64, device="cuda")
    lse = torch.zeros((B, Hq, S), dtype=torch.float64, device="cuda")
    d = torch.zeros((B, S, Hq + 2 * Hkv, D), dtype=torch.float64, device="cuda")
    step = max(1, min(S, (1 << 26) // S))
    for b in range(B):
        n = S if kv_len is None else int(kv_len[b])
        for h in range(Hq):
            kh = h // g
            x = qkv[b].reshape(S, Hq + 2 * Hkv, D)
            k, v = x[:n, Hq + kh].double(), x[:n, Hq + Hkv + kh].double()
            for i0 in range(0, S, step):
                i1 = min(S, i0 + step)
                m = min(n, i1) if case["causal"] else n
                q = x[i0:i1, h].double()
                s = (q @ k[:m].T).mul_(scale)
                if case["causal"]:
                    at = torch.arange(i0, i1, device="cuda")[:, None] < torch.arange(m, device="cuda")[None, :]
                    s.masked_fill_(at, -math.inf)
                L = torch.logsumexp(s, 1)
                p = s.sub_(L[:, None]).exp_()
                o[b, i0:i1, h], lse[b, h, i0:i1] = p @ v[:m], L
                if not case["bwd"]:
                    continue
                do = dout[b, i0:i1].reshape(i1 - i0, Hq, D)[:, h].double()
                d[b, :m, Hq + Hkv + kh] += p.T @ do
                ds = (do @ v[:m].T).sub_((do * o[b, i0:i1, h]).sum(1, keepdim=True)).mul_(p).mul_(scale)
                d[b, i0:i1, h] = ds @ k[:m]
                d[b, :m, Hq + kh] += ds.T @ q
    out = {"o": o.reshape(B, S, Hq * D), "lse": lse}
    if case["bwd"]:
        out["dqkv"] = d.reshape(B, S, -1)
    return out


def _rope(x, S, D, theta):
    """x [rows, heads, D]: pairs (2i, 2i+1) turned by pos * theta^(-i/D)."""
    i = torch.arange(D // 2, dtype=torch.float64, device=x.device)
    a = (torch.arange(x.shape[0], device=x.device) % S).double()[:, None] * torch.exp(-math.log(theta) * i / D)
    c, s = a.cos()[:, None], a.sin()[:, None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack((u * c - v * s, u * s + v * c), -1).reshape(x.shape)


def _rms(x, w, eps):
    """RMSNorm as the registry defines it: sums over aligned 64-channel groups, divided by C."""
    C = x.shape[1]
    t = x.reshape(x.shape[0], -1, min(C, 64))
    istd = torch.rsqrt(t.square().sum(2, keepdim=True) / C + eps)
    return (t * istd).reshape(x.shape) * w


def _exact_layer(case, seed):
    t = {k: v.double().requires_grad_() for k, v in _layer_inputs(case, seed).items()}
    Hq, Hkv, D, S, rows = case["Hq"], case["Hkv"], case["D"], case["S"], case["B"] * case["S"]
    nh, xhat, istd = Hq + Hkv, None, None
    v = _heads(t["x"] + t["bias"], Hq + 2 * Hkv, D)
    qk = v[:, :nh]
    if case["qknorm"]:
        istd = torch.rsqrt(qk.square().sum(2) / D + 1e-5)
        xhat = qk * istd[..., None]
        qk = xhat * _heads(t["gamma"][None], nh, D)
        xhat = xhat.reshape(rows, -1)
    if case["rope"]:
        qk = _rope(qk, S, D, 10000.0)
    qkv = torch.cat((qk, v[:, nh:]), 1).reshape(rows, -1)
    qkv.backward(t["dx"].detach())
    norm = _rms(t["h"] + t["res"], t["w"], float(np.float32(1e-5)))
    norm.backward(t["dh"].detach())
    F = case["F"]
    ffn = torch.nn.functional.silu(t["gu"][:, :F]) * t["gu"][:, F:]
    ffn.backward(t["df"].detach())
    keep = lambda x: None if x is None else x.detach()  # noqa: E731
    return {"qkv": qkv.detach(), "xhat": keep(xhat), "istd": keep(istd), "din": t["x"].grad,
            "dgamma": t["gamma"].grad if case["qknorm"] else None, "dbias": t["bias"].grad, "norm": norm.detach(),
            "dh": t["h"].grad, "dres": t["res"].grad, "dw": t["w"].grad, "ffn": ffn.detach(), "dgu": t["gu"].grad}


def _exact_model(case, seed):
    _, nodes = _graph(case)
    S, rows, ps = case["S"], case["B"] * case["S"], _params(nodes)
    ws = [w.double().requires_grad_(case["kind"] == "step") for w in _weights(case, nodes, seed)]
    of = {(n["id"], kind): w for (n, kind, _), w in zip(ps, ws)}
    x, y = _model_inputs(case, nodes, seed)
    act = {0: x.double()}

    def chain(ids, v):
        for i in ids:
            v = v + of[(i, "bias")] if nodes[i]["op"] == OP_BIAS else torch.nn.functional.silu(v)
        return v

    loss = top = None
    for n in nodes[1:]:
        if n["dead"]:
            continue
        i, op, v = n["id"], n["op"], act[n["in0"]]
        if op in GEMM:
            v = v @ of[(i, "W")]
        elif op == OP_RMSNORM:
            v = _rms(v, of[(i, "w")], n["fval"])
        elif op == OP_BIAS:
            v = v + of[(i, "bias")]
        elif op == OP_ADD:
            v = v + act[n["in1"]]
        elif op == OP_MUL:
            half = v.shape[1] // 2
            v = chain(n["left"], v[:, :half]) * chain(n["right"], v[:, half:])
        elif op == OP_PREP:
            nh, D = n["q_heads"] + n["kv_heads"], n["head_dim"]
            v = _heads(v + of[(i, "bias")], nh + n["kv_heads"], D)
            v = torch.cat((_rope(v[:, :nh], S, D, n["rope_theta"]), v[:, nh:]), 1).reshape(rows, -1)
        elif op == OP_GQA:
            Hq, Hkv, D = n["q_heads"], n["kv_heads"], n["head_dim"]
            v = v.reshape(case["B"], S, Hq + 2 * Hkv, D).transpose(1, 2)
            q, k, u = v[:, :Hq], v[:, Hq:Hq + Hkv], v[:, Hq + Hkv:]
            k, u = (z.repeat_interleave(Hq // Hkv, 1) for z in (k, u))
            s = (q @ k.transpose(2, 3)) / math.sqrt(D)
            s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1), -math.inf)
            v = (s.softmax(3) @ u).transpose(1, 2).reshape(rows, -1)
        elif op == OP_CE:
            loss = torch.nn.functional.cross_entropy(top, y.long())
            continue
        act[i] = top = v
    if case["kind"] == "infer":
        return {"logits": top.reshape(-1)}
    loss.backward()
    out = {}
    for k in _returned(nodes):           # one step of momentum SGD (Nesterov form) from rest
        w = ws[k].detach()
        g = ws[k].grad + (DECAY * w if ps[k][1] == "W" else 0)
        out["p%d" % k] = w - LR * (MOMENTUM * g + g)
    if case["host"]:
        out["loss"] = loss.detach()
    return out


def exact(case, seed):
    """What run() returns for these inputs, in 64 bits."""
    if case["kind"] == "attn":
        return _exact_attn(case, seed)
    return _exact_layer(case, seed) if case["kind"] == "layer" else _exact_model(case, seed)
