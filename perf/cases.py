"""The calls this framework is timed on: each kind of call a program makes through its public entry
points, at sizes from single-token decode to packed prefill and training, with 64-bit results to
compare with.

A case is a dict of plain values; `kind` names the call:

  decode_pool   StateSlotPool.fused_decode_step: one token for each of B sessions from raw projections
  decode_loop   GLADecodeGraphRunner.replay: `steps` decode steps of B sessions in one captured graph
  prefill_raw   fused_qkv_g_prep_chunk_gla: VectorisedGLA's prefill from raw projections
  prefill       fast_chunk_gla without gradients
  packed        fast_chunk_gla_varlen over n ragged sequences with per-sequence states
  gdn           fast_chunk_gated_deltanet without gradients
  gla_train     fast_chunk_gla forward and backward
  gdn_train     fast_chunk_gated_deltanet forward and backward

Gates: "key" is one log-decay per key dim, "head" one per (token, head).  Distributions are those of
triune_amd.workloads: q scaled by D^-1/2, k, v ~ N(0, 1), g = logsigmoid(N(0, 1)) / 16 for GLA; Gated
DeltaNet takes L2-normalised q and k, and either the mild per-head decay exp(-softplus / 8) with a
per-head beta, or the reference model's per-key-dim logsigmoid gates without beta.
"""

from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from triune_amd import fast_chunk_gated_deltanet, fast_chunk_gla, fast_chunk_gla_varlen, fused_qkv_g_prep_chunk_gla
from triune_amd.serving import GLADecodeGraphRunner, StateSlotPool

DEV = "cuda"
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # one session generating a token: the smallest call, all latency (H = 8, head dim 64: d = 512)
        {"name": "decode_one", "kind": "decode_pool", "B": 1, "H": 8, "D": 64, "io": "bf16"},
        # batched decode in the graph runner, 256 sessions of 6 heads
        {"name": "decode_loop", "kind": "decode_loop", "steps": 32, "B": 256, "H": 6, "D": 64, "io": "bf16"},
        # VectorisedGLA's 1024-token prefill tile, pre-processing included
        {"name": "prefill_tile", "kind": "prefill_raw", "B": 4, "T": 1024, "H": 6, "D": 64, "io": "bf16"},
        # long-context prefill over a carried-in state: the headline benchmark's shape
        {"name": "prefill_long", "kind": "prefill", "B": 4, "T": 16384, "H": 6, "D": 64, "io": "bf16", "gate": "bf16",
         "s0": True},
        # prompts of an odd length with the gate computed in fp32, as under autocast (d = 512)
        {"name": "prefill_odd", "kind": "prefill", "B": 3, "T": 3001, "H": 8, "D": 64, "io": "bf16", "gate": "fp32",
         "s0": False},
        # fp32 model, one prompt: the reference's CPU configuration on the GPU
        {"name": "prefill_fp32", "kind": "prefill", "B": 1, "T": 2048, "H": 6, "D": 64, "io": "fp32", "gate": "fp32",
         "s0": False},
        # continuous batching: 32 ragged prompts of 128 to 8192 tokens at d_model 1536
        {"name": "prefill_packed", "kind": "packed", "n": 32, "lo": 128, "hi": 8192, "lseed": 4, "H": 12, "D": 128,
         "io": "bf16"},
        # Gated DeltaNet prefill, one decay and one beta per token and head
        {"name": "gdn_prefill", "kind": "gdn", "B": 4, "T": 8192, "H": 6, "D": 64, "io": "bf16", "gate": "head",
         "beta": True},
        # Gated DeltaNet prefill as the reference model calls it: head dim 128, gates per key dim, no beta
        {"name": "gdn_prefill_wide", "kind": "gdn", "B": 4, "T": 8192, "H": 12, "D": 128, "io": "bf16", "gate": "key",
         "beta": False},
        # GLA training step of the recall benchmark (d = 256, 4 heads)
        {"name": "gla_train", "kind": "gla_train", "B": 8, "T": 2048, "H": 4, "D": 64, "io": "bf16"},
        # Gated DeltaNet training step, per-head decay and beta
        {"name": "gdn_train", "kind": "gdn_train", "B": 4, "T": 8192, "H": 6, "D": 64, "io": "bf16", "gate": "head",
         "beta": True},
        # Gated DeltaNet training step of the reference model: head dim 128, gates per key dim, no beta
        {"name": "gdn_train_wide", "kind": "gdn_train", "B": 4, "T": 2048, "H": 12, "D": 128, "io": "bf16",
         "gate": "key", "beta": False},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random):
    kind = rng.choice(["decode_pool", "decode_loop", "prefill_raw", "prefill", "prefill", "packed", "gdn", "gdn",
                       "gla_train", "gdn_train", "gdn_train"])
    io = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    D = rng.choice([64, 128])
    if kind == "decode_pool":
        return {"kind": kind, "B": _log(rng, 1, 256), "H": rng.choice([4, 6, 8, 12]), "D": D, "io": io}
    if kind == "decode_loop":
        return {"kind": kind, "steps": _log(rng, 4, 32), "B": _log(rng, 8, 256), "H": rng.choice([4, 6]), "D": 64,
                "io": io}
    if kind == "prefill_raw":
        return {"kind": kind, "B": rng.randint(1, 4), "T": _log(rng, 128, 16384), "H": rng.choice([4, 6, 8]), "D": 64,
                "io": io}
    if kind == "prefill":
        io = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        gate = rng.choice([io, "fp32"])
        T = _log(rng, 200, 16384 if io != "fp32" and D == 64 else 4096)
        return {"kind": kind, "B": rng.randint(1, 4), "T": T, "H": rng.choice([4, 6, 8, 12]), "D": D, "io": io,
                "gate": gate, "s0": rng.random() < 0.5}
    if kind == "packed":
        return {"kind": kind, "n": _log(rng, 2, 32), "lo": rng.randint(1, 128), "hi": _log(rng, 512, 8192),
                "lseed": rng.randrange(1000), "H": rng.choice([6, 8, 12]), "D": D, "io": io}
    gate, beta = rng.choice([("head", True), ("head", False), ("key", False), ("key", True)])
    if kind == "gdn":
        return {"kind": kind, "B": rng.randint(1, 4), "T": _log(rng, 100, 8192), "H": rng.choice([4, 6, 8, 12]), "D": D,
                "io": io, "gate": gate, "beta": beta}
    if kind == "gla_train":
        return {"kind": kind, "B": rng.randint(1, 8), "T": _log(rng, 100, 4096), "H": rng.choice([4, 6, 8]), "D": D,
                "io": io}
    return {"kind": kind, "B": rng.randint(1, 4), "T": _log(rng, 100, 8192 if D == 64 else 2048),
            "H": rng.choice([4, 6, 8, 12]), "D": D, "io": io, "gate": gate, "beta": beta}


# ---------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------


def _lengths(case):
    r = random.Random(case["lseed"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["n"])]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV)


def _gla_inputs(gen, lead, H, D, dt, gdt):
    q = (_randn(gen, *lead, H, D) * D**-0.5).to(dt)
    k, v = _randn(gen, *lead, H, D).to(dt), _randn(gen, *lead, H, D).to(dt)
    return q, k, v, (F.logsigmoid(_randn(gen, *lead, H, D)) / 16).to(gdt)


def _gdn_inputs(gen, case, dt):
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    q, k = (F.normalize(_randn(gen, B, T, H, D), dim=-1).to(dt) for _ in range(2))
    v = _randn(gen, B, T, H, D).to(dt)
    if case["gate"] == "head":
        g = (-F.softplus(_randn(gen, B, T, H)) / 8).to(dt)
    else:
        g = F.logsigmoid(_randn(gen, B, T, H, D)).to(dt)
    beta = torch.sigmoid(_randn(gen, B, T, H)).to(dt) if case["beta"] else None
    return q, k, v, g, beta


def _rope(T, D, at=0):
    inv = 1.0 / (10000.0 ** (torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D))
    a = torch.outer(torch.arange(at, at + T, device=DEV, dtype=torch.float64), inv).repeat(1, 2)
    return a.cos().float(), a.sin().float()


def _inputs(case, seed):
    """The call's tensors, from the seed alone."""
    kind, H, D, dt, gen = case["kind"], case["H"], case["D"], _DT[case["io"]], _gen(seed)
    if kind == "decode_pool":
        B = case["B"]
        states = 0.1 * _randn(gen, B, H, D, D)
        cos, sin = _rope(1, D, at=1000)
        return {"qkvg": _randn(gen, B, 4, H, D).to(dt), "states": states, "cos": cos, "sin": sin}
    if kind == "decode_loop":
        n, B = case["steps"], case["B"]
        q, k, v = (_randn(gen, n, B, H, D).to(dt) for _ in range(3))
        g = (F.logsigmoid(_randn(gen, n, B, H, D)) / 16).to(dt)
        return {"q": q, "k": k, "v": v, "g": g, "states": 0.1 * _randn(gen, B, H, D, D)}
    if kind == "prefill_raw":
        B, T = case["B"], case["T"]
        cos, sin = _rope(T, D)
        return {"qkv": _randn(gen, B, T, 3, H, D).to(dt), "g": _randn(gen, B, T, H, D).to(dt), "cos": cos, "sin": sin,
                "s0": 0.1 * _randn(gen, B, H, D, D)}
    if kind == "packed":
        lens = _lengths(case)
        q, k, v, g = _gla_inputs(gen, (1, sum(lens)), H, D, dt, dt)
        cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=DEV)
        return {"q": q, "k": k, "v": v, "g": g, "cu": cu, "s0": 0.1 * _randn(gen, len(lens), H, D, D)}
    B, T = case["B"], case["T"]
    if kind in ("prefill", "gla_train"):
        gdt = _DT[case["gate"]] if kind == "prefill" else dt
        q, k, v, g = _gla_inputs(gen, (B, T), H, D, dt, gdt)
        s0 = 0.1 * _randn(gen, B, H, D, D) if case.get("s0") else None
        s = {"q": q, "k": k, "v": v, "g": g, "s0": s0}
    else:
        q, k, v, g, beta = _gdn_inputs(gen, case, dt)
        s = {"q": q, "k": k, "v": v, "g": g, "beta": beta}
    if kind.endswith("_train"):
        s["do"] = _randn(gen, B, T, H, D).to(dt)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind, B = case["kind"], case.get("B")
    s["kind"] = kind
    if kind == "decode_pool":
        pool = StateSlotPool(1, B, case["H"], case["D"], case["D"], device=DEV)
        s["slots"] = pool.slots_tensor([f"session {i}" for i in range(B)])
        pool.states[0, s["slots"].long()] = s.pop("states")
        s["pool"] = pool
    elif kind == "decode_loop":
        slots = torch.arange(B, device=DEV, dtype=torch.int32)
        runner = GLADecodeGraphRunner(s["states"], slots, steps=case["steps"], dtype=_DT[case["io"]])
        for name in "qkvg":
            getattr(runner, name).copy_(s.pop(name))
        runner.capture()
        s["runner"] = runner
    elif kind.endswith("_train"):
        s["leaves"] = [x.requires_grad_() for x in (s["q"], s["k"], s["v"], s["g"], s.get("beta")) if x is not None]
    return s


def run(s):
    kind = s["kind"]
    if kind == "decode_pool":
        o = s["pool"].fused_decode_step(0, s["qkvg"], s["slots"], s["cos"], s["sin"])
        return o, s["pool"].states, s["pool"].offsets
    if kind == "decode_loop":
        return s["runner"].replay(), s["states"]
    if kind == "prefill_raw":  # in place, as the reference: q and k are replaced and the outputs go over g
        o, st = fused_qkv_g_prep_chunk_gla(s["qkv"], s["g"], s["cos"], s["sin"], initial_state=s["s0"])
        return o, st, s["qkv"]
    if kind == "prefill":
        return fast_chunk_gla(s["q"], s["k"], s["v"], s["g"], initial_state=s["s0"])
    if kind == "packed":
        return fast_chunk_gla_varlen(s["q"], s["k"], s["v"], s["g"], s["cu"], initial_state=s["s0"])
    if kind == "gdn":
        return fast_chunk_gated_deltanet(s["q"], s["k"], s["v"], s["g"], beta=s["beta"])
    if kind == "gla_train":
        o, st = fast_chunk_gla(s["q"], s["k"], s["v"], s["g"])
    else:
        o, st = fast_chunk_gated_deltanet(s["q"], s["k"], s["v"], s["g"], beta=s["beta"])
    return (o.detach(), st.detach(), *torch.autograd.grad(o, s["leaves"], s["do"]))


def work(case):
    kind, H, D = case["kind"], case["H"], case["D"]
    io = _DT[case["io"]].itemsize
    state = H * D * D * 4
    if kind in ("decode_pool", "decode_loop"):
        # every step reads and writes the states: in a model the next step's inputs depend on its output
        n = case["B"] * case.get("steps", 1)
        return {"bytes": n * (2 * state + 5 * H * D * io), "flops": n * 5 * H * D * D}
    N = sum(_lengths(case)) if kind == "packed" else case["B"] * case["T"]
    nseq = case["n"] if kind == "packed" else case["B"]
    gla = 2 * (2 * 64 * D + 2 * D * D)  # flops per token-head of 64-token chunks
    gdn = 2 * (4 * 64 * D + 3 * D * D)
    if kind == "prefill_raw":  # q, k, g, v in; q, k and the outputs (over g) out
        return {"bytes": N * H * D * 7 * io + 2 * nseq * state + 2 * case["T"] * D * 4, "flops": N * H * gla}
    if kind in ("prefill", "packed"):
        gb = _DT[case["gate"]].itemsize if kind == "prefill" else io
        states = 2 if kind == "packed" or case["s0"] else 1
        return {"bytes": N * H * D * (4 * io + gb) + states * nseq * state, "flops": N * H * gla}
    if kind == "gla_train":  # q, k, v, g, do in; o, dq, dk, dv, dg out
        return {"bytes": N * H * D * 10 * io + nseq * state, "flops": 3 * N * H * gla}
    per_token = (D if case["gate"] == "key" else 1) + (1 if case["beta"] else 0)
    if kind == "gdn":
        return {"bytes": N * H * (4 * D + per_token) * io + nseq * state, "flops": N * H * gdn}
    return {"bytes": N * H * (8 * D + 2 * per_token) * io + nseq * state, "flops": 3 * N * H * gdn}


# About four times the error of each output type against exact(): bf16 outputs are 1.7e-3 off by their
# own rounding (a sum of rounded gradients 2.4e-3), fp16 ones an eighth of that, fp32 ones 2e-7 to 1e-6.
_REL = {"bf16": 8e-3, "fp16": 1.5e-3, "fp32": 4e-6}


def tolerance(case):
    return {"rel": _REL[case["io"]]}


# ---------------------------------------------------------------------------------------
# Results in 64 bits: the recurrences token by token
# ---------------------------------------------------------------------------------------


def _scan(q, k, v, g, beta, S, delta):
    """q, k, v [B, T, H, D], g [B, T, H, D or 1], beta [B, T, H] or None, float64: outputs and final state of
    S <- diag(exp(g)) S + beta k u^T, o = S^T q, with u = v (GLA) or v - S^T k before the decay."""
    a = g.exp().unsqueeze(-1)
    w = k if beta is None else k * beta.unsqueeze(-1)
    out = []
    for t in range(q.shape[1]):
        u = v[:, t]
        if delta:
            u = u - (S * k[:, t].unsqueeze(-1)).sum(-2)
        S = a[:, t] * S + w[:, t].unsqueeze(-1) * u.unsqueeze(-2)
        out.append((S * q[:, t].unsqueeze(-1)).sum(-2))
    return torch.stack(out, 1), S


def _grads(ins, S0, do, delta, seg=128):
    """Outputs, final state and the gradients of `ins` (q, k, v, g, beta) for upstream do: autograd
    over segments of the recurrence, last to first."""
    T = do.shape[1]

    def part(t):
        q, k, v, g, beta = (None if x is None else x[:, t:t + seg] for x in ins)
        return q, k, v, g.clamp(max=0), beta

    starts, outs, S = [], [], S0
    with torch.no_grad():
        for t in range(0, T, seg):
            starts.append(S)
            o, S = _scan(*part(t), S, delta)
            outs.append(o)
    grads, dS = [], torch.zeros_like(S0)
    for i, t in reversed(list(enumerate(range(0, T, seg)))):
        leaf = [None if x is None else x[:, t:t + seg].clone().requires_grad_() for x in ins]
        s = starts[i].clone().requires_grad_()
        o, e = _scan(leaf[0], leaf[1], leaf[2], leaf[3].clamp(max=0), leaf[4], s, delta)
        on = [x for x in leaf if x is not None]
        got = torch.autograd.grad([o, e], on + [s], [do[:, t:t + seg], dS])
        grads.append(got[:-1])
        dS = got[-1]
    grads = [torch.cat(x, 1) for x in zip(*reversed(grads))]
    return (torch.cat(outs, 1), S, *grads)


def _prep(x, cos, sin):
    """RoPE(normalize(elu(x) + 1)) over the last dim."""
    x = F.elu(x) + 1
    x = x / x.square().sum(-1, keepdim=True).clamp_min(1e-12).sqrt()
    a, b = x.chunk(2, dim=-1)
    return x * cos + torch.cat([-b, a], dim=-1) * sin


def exact(case, seed):
    s = {n: x.double() if torch.is_tensor(x) and x.is_floating_point() else x for n, x in _inputs(case, seed).items()}
    kind, H, D = case["kind"], case["H"], case["D"]
    if kind == "decode_pool":
        q, k, v, g = s["qkvg"].unbind(1)
        q, k = (_prep(x, s["cos"], s["sin"]).unsqueeze(1) for x in (q, k))
        o, S = _scan(q, k, v.unsqueeze(1), F.logsigmoid(g).unsqueeze(1), None, s["states"], False)
        return o, S.unsqueeze(0), None
    if kind == "decode_loop":
        o, S = _scan(*(s[n].transpose(0, 1) for n in "qkvg"), None, s["states"], False)
        return o.transpose(0, 1), S
    if kind == "prefill_raw":
        q, k, v = s["qkv"].unbind(2)
        cos, sin = s["cos"].unsqueeze(1), s["sin"].unsqueeze(1)
        q, k = _prep(q, cos, sin), _prep(k, cos, sin)
        o, S = _scan(q, k, v, F.logsigmoid(s["g"]), None, s["s0"], False)
        return o, S, torch.stack([q, k, v], 2)
    if kind == "packed":  # sequences side by side, padded at their end with tokens that change nothing
        lens = _lengths(case)
        n, T = len(lens), max(lens)
        pad = {m: torch.zeros(n, T, H, D, device=DEV, dtype=torch.float64) for m in "qkvg"}
        cu = s["cu"].tolist()
        for i, (a, b) in enumerate(zip(cu, cu[1:])):
            for m in "qkvg":
                pad[m][i, :b - a] = s[m][0, a:b]
        o, S = _scan(*(pad[m] for m in "qkvg"), None, s["s0"], False)
        return torch.cat([o[i, :ln] for i, ln in enumerate(lens)]).unsqueeze(0), S
    S0 = s.get("s0")
    if S0 is None:
        S0 = torch.zeros(case["B"], H, D, D, device=DEV, dtype=torch.float64)
    if kind == "prefill":
        return _scan(s["q"], s["k"], s["v"], s["g"].clamp(max=0), None, S0, False)
    head = kind.startswith("gdn") and case["gate"] == "head"
    ins = [s["q"], s["k"], s["v"], s["g"].unsqueeze(-1) if head else s["g"], s.get("beta")]
    if kind == "gdn":
        return _scan(*ins[:3], ins[3].clamp(max=0), ins[4], S0, True)
    got = list(_grads(ins, S0, s["do"], kind == "gdn_train"))
    if head:
        got[5] = got[5].squeeze(-1)
    return tuple(got)
