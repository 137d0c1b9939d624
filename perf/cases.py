"""The framework's work as a user's program asks for it: decode steps, prefill
and training steps of the delta-rule recurrence, through the package's public
entry points.

A case is a dict of plain values:

  op         "step" (one decode token), "steps" (T tokens in one launch),
             "prefill", "stream" (prefill in token blocks, fused prologue), "train"
  variant    "gdn2", "gdn", "kda", "gla" or "delta"
  B, L       batch rows and tokens per row (decode: L tokens per call)
  Hk, Hv     key and value heads (K = V = 128, the only size the API takes)
  dtype      q/k/v: "bf16" or "f32"
  precision  the entry point's ``precision`` (prefill and training)
  state      decode: the carried state's type, "bf16" or "f32"
  doc        mean document length of packed rows, 0 for one document
  init       prefill: starts from a carried state
  reset      decode: a reset flag per row is passed
  recompute  training: ``recompute_states``

``prepare`` makes the inputs on the GPU from the seed, ``run`` is one call (one
forward and backward in training), ``exact`` is the token-by-token recurrence in
float64 with torch alone.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "deltanet-tpu_amd"))

from deltanet_tpu_amd import (  # noqa: E402
    chunk_delta_rule, chunk_gdn, chunk_gdn2, chunk_gla, chunk_kda, delta_rule_decode_step, gdn2_decode_step,
    gdn2_decode_steps, gdn_decode_step, gla_decode_step, kda_decode_step)

D = 128
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
CHUNKED = {"gdn2": chunk_gdn2, "gdn": chunk_gdn, "kda": chunk_kda, "gla": chunk_gla, "delta": chunk_delta_rule}
STEP = {"gdn2": gdn2_decode_step, "gdn": gdn_decode_step, "kda": kda_decode_step, "gla": gla_decode_step,
        "delta": delta_rule_decode_step}
GATES = {"gdn2": ("g", "b", "w"), "gdn": ("g", "beta"), "kda": ("g", "beta"), "gla": ("g",), "delta": ("beta",)}


def _case(op, variant, B, L, Hk, Hv, dtype="bf16", precision="bf16", state="f32", doc=0, init=False, reset=False,
          recompute=False):
    return dict(op=op, variant=variant, B=B, L=L, Hk=Hk, Hv=Hv, dtype=dtype, precision=precision, state=state, doc=doc,
                init=init, reset=reset, recompute=recompute)


def listed():
    c = _case
    return [
        # one user's token: a single sequence, 16 key and 32 value heads, state stored in 16 bits
        dict(c("step", "gdn2", 1, 1, 16, 32, state="bf16"), name="step-1"),
        # a small serving batch of the scalar-decay layer, float32 state, some rows starting over
        dict(c("step", "gdn", 32, 1, 16, 32, state="f32", reset=True), name="gdn-step-32"),
        # a full serving batch: the state (268 MB in 16 bits) read and written once
        dict(c("step", "gdn2", 256, 1, 16, 32, state="bf16"), name="step-256"),
        # a draft of 16 tokens verified, or a prompt's short tail, for 64 sequences
        dict(c("steps", "gdn2", 64, 16, 16, 32, state="bf16"), name="steps-64x16"),
        # the rest of a prompt after a cached prefix: short, ragged, from a carried state
        dict(c("prefill", "gdn2", 1, 300, 12, 24, init=True), name="prefill-300"),
        # an ordinary prompt with two documents, channel-wise gates
        dict(c("prefill", "gdn2", 1, 2048, 12, 24, doc=1024), name="prefill-2048"),
        # float32 throughout, ragged, one value head per key head
        dict(c("prefill", "kda", 2, 1000, 16, 16, dtype="f32", precision="fp32"), name="kda-prefill-fp32"),
        # a large batch of packed documents through the scalar-decay layer
        dict(c("prefill", "gdn", 4, 8192, 16, 32, doc=1024), name="gdn-prefill-4x8192"),
        # a long context in blocks of 8192 tokens, raw gates
        dict(c("stream", "gdn2", 1, 65536, 16, 32, doc=8192), name="stream-65536"),
        # training at the ordinary prompt's size, and packed rows through the scalar-decay layer
        dict(c("train", "gdn2", 1, 2048, 12, 24, doc=1024), name="train-2048"),
        dict(c("train", "gdn", 1, 4096, 16, 32, doc=1024), name="gdn-train-4096"),
        # training in float32 at a ragged length
        dict(c("train", "kda", 2, 777, 8, 8, dtype="f32", precision="fp32"), name="kda-train-fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["step", "steps", "prefill", "prefill", "stream", "train", "train"])
    variant = rng.choice(list(CHUNKED))
    # as many value heads as key heads, or a group of them per key head
    Hk, Hv = rng.choice([(2, 4), (12, 24), (16, 32), (16, 16), (8, 32)])
    dtype, precision = rng.choice([("bf16", "bf16"), ("bf16", "bf16"), ("f32", "bf16"), ("f32", "fp32")])
    if op == "step":
        return _case(op, variant, _log_int(rng, 1, 256), 1, Hk, Hv, dtype=dtype, state=rng.choice(["bf16", "f32"]),
                     reset=rng.random() < 0.5)
    if op == "steps":
        return _case(op, "gdn2", _log_int(rng, 1, 256), rng.randint(2, 32), Hk, Hv, dtype=dtype,
                     state=rng.choice(["bf16", "f32"]), reset=rng.random() < 0.5)
    if op == "stream":
        return _case(op, "gdn2", 1, _log_int(rng, 8193, 60000), Hk, Hv, doc=rng.choice([0, 2048, 8192]))
    most = 8192 if op == "train" else 32768
    most = most // 2 if dtype == "f32" else most
    B = rng.choice([1, 1, 2, 3, 4, 8])
    L = _log_int(rng, 16, min(most // B, 4096 if op == "train" else 16384))
    return _case(op, variant, B, L, Hk, Hv, dtype=dtype, precision=precision, doc=rng.choice([0, 0, 128, 1024]),
                 init=op == "prefill" and rng.random() < 0.3, recompute=op == "train" and rng.random() < 0.3)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _documents(seed, B, L, mean):
    """segment_ids of packed rows: document lengths geometric with this mean, at least 16 tokens."""
    rng = np.random.default_rng(seed)
    seg = np.zeros((B, L), np.int32)
    for b in range(B):
        t, d = 0, 0
        while t < L:
            n = int(max(rng.geometric(1.0 / mean), 16))
            seg[b, t:t + n] = d
            t, d = t + n, d + 1
    return torch.from_numpy(seg).cuda()


def _gates(case, rn, rand):
    """The variant's gates with the distributions of the layers that produce them."""
    B, L, Hk, Hv = case["B"], case["L"], case["Hk"], case["Hv"]
    v = case["variant"]
    if case["op"] == "stream":  # pre-activation values; the prologue activates them
        return {"g": rn(B, L, Hk, D), "b": rn(B, L, Hk, D), "w": rn(B, L, Hv, D)}
    if v == "gdn":  # one decay and one beta per token and value head: -A softplus(a), sigmoid
        a = torch.exp(math.log(16.0) * rand(Hv))
        return {"g": -a * torch.nn.functional.softplus(rn(B, L, Hv)), "beta": torch.sigmoid(rn(B, L, Hv))}
    gates = {}
    if v != "delta":
        gates["g"] = -torch.exp(0.39 * rn(B, L, Hk, D) - 1.0)
    if v == "gdn2":
        gates["b"] = torch.sigmoid(0.39 * rn(B, L, Hk, D))
        gates["w"] = torch.sigmoid(0.39 * rn(B, L, Hv, D))
    elif v != "gla":
        gates["beta"] = torch.sigmoid(rn(B, L, Hk))
    return gates


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    rand = lambda *s: torch.rand(*s, device="cuda", generator=gen)
    B, L, Hk, Hv, dt = case["B"], case["L"], case["Hk"], case["Hv"], DTYPES[case["dtype"]]
    s = {"case": case, "q": rn(B, L, Hk, D).to(dt), "k": rn(B, L, Hk, D).to(dt), "v": rn(B, L, Hv, D).to(dt)}
    s.update(_gates(case, rn, rand))
    if case["op"] in ("step", "steps"):
        s["state"] = (0.02 * rn(B, Hv, D, D)).to(DTYPES[case["state"]])
        s["reset"] = rand(B) < 0.1 if case["reset"] else None
        return s
    s["seg"] = _documents(seed, B, L, case["doc"]) if case["doc"] else None
    s["init"] = 0.1 * rn(B, Hv, D, D) if case["init"] else None
    if case["op"] == "train":
        s["d_out"] = rn(B, L, Hv, D).to(dt)
        s["leaves"] = [s[n].requires_grad_(True) for n in ("q", "k", "v") + GATES[case["variant"]]]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    c = s["case"]
    gates = [s[n] for n in GATES[c["variant"]]]
    if c["op"] == "step":
        return STEP[c["variant"]](s["q"], s["k"], s["v"], *gates, s["state"], reset=s["reset"], qk_l2norm=True,
                                  state_dtype=DTYPES[c["state"]])
    if c["op"] == "steps":
        return gdn2_decode_steps(s["q"], s["k"], s["v"], *gates, s["state"], reset=s["reset"], qk_l2norm=True,
                                 state_dtype=DTYPES[c["state"]])
    f = CHUNKED[c["variant"]]
    if c["op"] == "train":
        out = f(s["q"], s["k"], s["v"], *gates, segment_ids=s["seg"], qk_l2norm=True, precision=c["precision"],
                recompute_states=c["recompute"])
        return [out.detach(), list(torch.autograd.grad(out, s["leaves"], s["d_out"]))]
    stream = dict(fuse_prologue=True, streaming_prefill=True, prefill_block_size=8192) if c["op"] == "stream" else {}
    return f(s["q"], s["k"], s["v"], *gates, segment_ids=s["seg"], initial_state=s["init"], output_final_state=True,
             qk_l2norm=True, is_inference=True, precision=c["precision"], **stream)


def work(case):
    """Inputs read once, outputs written once; the recurrence's own operations per
    token and value head: decay, S^T(b k), the rank-one update and S^T q are 7
    operations per state element (three times that forward and backward)."""
    B, L, Hk, Hv, op, v = case["B"], case["L"], case["Hk"], case["Hv"], case["op"], case["variant"]
    e, n = (2 if case["dtype"] == "bf16" else 4), B * L
    qkv = n * D * e * (2 * Hk + Hv)
    gates = 4 * n * {"gdn2": 2 * Hk * D + Hv * D, "gdn": 2 * Hv, "kda": Hk * D + Hk, "gla": Hk * D, "delta": Hk}[v]
    out = n * D * e * Hv
    state = B * Hv * D * D * (2 if op in ("step", "steps") and case["state"] == "bf16" else 4)
    flops = 7.0 * n * Hv * D * D
    if op == "train":  # inputs read by both directions, the output's gradient read, all gradients written
        return {"bytes": 3.0 * (qkv + gates) + 2.0 * out, "flops": 3.0 * flops}
    states = 2 if op in ("step", "steps") or case["init"] else 1
    seg = 4 * n if case["doc"] else 0
    return {"bytes": float(qkv + gates + out + states * state + seg), "flops": flops}


def tolerance(case):
    """About four times what the listed and forty drawn cases were off the float64
    recurrence (largest rel / max seen): decode 1.7e-3 / 3.9e-3 with a 16-bit output
    or state (one rounding) and 3.4e-7 / 3.0e-6 in float32; precision "bf16"
    2.6e-3 / 1.5e-2; precision "fp32" 8.6e-7 / 1.3e-5."""
    decode = case["op"] in ("step", "steps")
    if decode and (case["dtype"] == "bf16" or case["state"] == "bf16"):
        return {"rel": 7e-3, "max": 1.6e-2}
    if decode or case["precision"] == "fp32":
        return {"rel": 4e-6, "max": 5e-5}
    return {"rel": 1e-2, "max": 6e-2}


# ---------------------------------------------------------------------------
# the recurrence in float64
# ---------------------------------------------------------------------------

class _Round(torch.autograd.Function):
    """A value as its 16-bit type holds it; the gradient passes."""

    @staticmethod
    def forward(ctx, x, dt):
        return x.to(dt).to(torch.float64)

    @staticmethod
    def backward(ctx, g):
        return g, None


def _tokens(S, q, k, v, a, b, keep):
    """Some tokens of the recurrence: q, k, b (T, B, H, 128); v = w v; a the decay; keep (T, B) 0 where a document starts."""
    out = []
    for t in range(q.shape[0]):
        S = S * (a[t] if keep is None else a[t] * keep[t][:, None, None])[..., None]
        u = v[t] - torch.matmul(b[t][..., None, :], S)[..., 0, :]
        S = S + k[t][..., None] * u[..., None, :]
        out.append(torch.matmul(q[t][..., None, :], S)[..., 0, :])
    return torch.stack(out), S


def _scan(case, x, seg, S):
    """Output (B, L, Hv, 128) and last state for float64 inputs `x` of the entry point."""
    B, L, Hk, Hv, v = case["B"], case["L"], case["Hk"], case["Hv"], case["variant"]
    one = torch.ones((B, L, 1, 1), dtype=torch.float64, device="cuda")
    four = lambda t: t if t.ndim == 4 else t[..., None]
    g = four(x["g"]) if "g" in x else 0.0 * one
    b = four(x["b"] if "b" in x else x["beta"]) if v != "gla" else 0.0 * one
    w = four(x["w"] if "w" in x else x["beta"]) if v != "gla" else one
    if case["op"] == "stream":
        g, b, w = -torch.exp(torch.clamp(g, max=5.0)), torch.sigmoid(b), torch.sigmoid(w)
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    q, k = unit(x["q"]) / math.sqrt(D), unit(x["k"])
    if case["dtype"] == "bf16" and case["op"] in ("prefill", "train"):  # normalised rows are kept in the input's type
        q, k = _Round.apply(q, torch.bfloat16), _Round.apply(k, torch.bfloat16)
    # time first, every operand at the value heads
    heads = lambda t: (t if t.shape[2] in (1, Hv) else t.repeat_interleave(Hv // Hk, dim=2)).transpose(0, 1)
    q, k, b, w, a = heads(q), heads(k), heads(b), heads(w), heads(torch.exp(g))
    wv, b = w * x["v"].transpose(0, 1), b * k
    keep = None
    if seg is not None:
        keep = torch.ones((L, B), dtype=torch.float64, device="cuda")
        keep[1:] = (seg[:, 1:] == seg[:, :-1]).to(torch.float64).T
    outs, n = [], 64
    for t in range(0, L, n):
        part = (S,) + tuple(y[t:t + n] for y in (q, k, wv, a, b)) + (None if keep is None else keep[t:t + n],)
        if case["op"] == "train":  # keeps one state in 64 for the way back
            o, S = torch.utils.checkpoint.checkpoint(_tokens, *part, use_reentrant=False)
        else:
            o, S = _tokens(*part)
        outs.append(o)
    return torch.cat(outs).transpose(0, 1), S


def exact(case, seed):
    s = prepare(case, seed)
    names = ("q", "k", "v") + GATES[case["variant"]]
    x = {n: s[n].detach().to(torch.float64) for n in names}
    B, Hv, op = case["B"], case["Hv"], case["op"]
    S = s.get("state") if op in ("step", "steps") else s["init"]
    S = torch.zeros((B, Hv, D, D), dtype=torch.float64, device="cuda") if S is None else S.to(torch.float64)
    if s.get("reset") is not None:
        S = torch.where(s["reset"][:, None, None, None], torch.zeros_like(S), S)
    if op == "train":
        for n in names:
            x[n].requires_grad_(True)
        out, _ = _scan(case, x, s["seg"], S)
        return [out.detach(), list(torch.autograd.grad(out, [x[n] for n in names], s["d_out"].to(torch.float64)))]
    with torch.no_grad():
        out, S = _scan(case, x, s.get("seg"), S)
    return out, S
