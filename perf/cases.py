"""The workloads by which the operator's speed is judged: what a program that
serves or trains hybrid Gated DeltaNet layers has this package do, through its
public entry points.

Five kinds of call, each over the whole range of its sizes:

  decode   one token of each running request through the layer
           (decode_layer_step) against slot pools of conv tails and states
  verify   a few drafted tokens per request, every state kept in a slot of its
           own (recurrent_fwd with token_state_idx), speculative decoding
  prefill  the operator by itself, as the reference's API calls it
           (gated_delta_rule): one long sequence, batches, packed sequences
  layer    a serving engine's prefill batch through the layer: packed requests,
           convolution, norms and gates (layer_prologue_varlen), then the
           operator against state slots with the epilogue (chunk_layer_fwd_slots)
  train    the operator's forward and backward through autograd

Head shapes are those of the repository's workloads: 16 key heads for 32 value
heads of width 128, four heads of width 64 in float32 (the small prefill), and
the 256-wide heads. Gates follow the layer's own parameters (A uniform in
(0, 16), dt_bias around -4), so decays run from almost none to strong across
the heads.

A case is a dict of plain values:
  kind, dtype (of q, k, v or of the projection), hk, hv, dk, dv,
  batch, length   (decode, verify, and unpacked prefill and train)
  seqs, tokens    (packed: that many sequences of uneven lengths, in all `tokens`)
  state           dtype of the state pool (decode, verify, layer)
  tail            dtype of the conv tail pool (decode, layer)
  out             dtype of the layer's output (decode, layer)
  l2norm          normalisation of q and k (decode, layer)
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from pseudobrain_amd.gated_deltanet import gated_delta_rule, recurrent_fwd
from pseudobrain_amd.layer import chunk_layer_fwd_slots, decode_layer_step, layer_prologue_varlen

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
WIDE = dict(hk=16, hv=32, dk=128, dv=128)   # the Qwen3-Next layer's heads
SMALL = dict(hk=4, hv=4, dk=64, dv=64)      # the reference's small float32 prefill
K256 = dict(hk=16, hv=32, dk=256, dv=256)   # the widest heads the device gate admits
CONV = 4
EPS = 1e-5
CHUNK = 64


def _case(kind, dtype="bfloat16", heads=None, **sizes):
    return dict(kind=kind, dtype=dtype, **(WIDE if heads is None else heads), **sizes)


def listed():
    served = dict(tail="bfloat16", l2norm="max")
    return [
        # one user at the keyboard: a single request's next token, latency only
        dict(_case("decode", batch=1, state="bfloat16", out="bfloat16", **served), name="decode_b1"),
        # a steady serving batch, states kept in float32
        dict(_case("decode", batch=64, state="float32", out="bfloat16", **served), name="decode_b64"),
        # a full serving batch of an odd size, states in the model's dtype, the model's own q/k norm
        dict(_case("decode", batch=233, state="bfloat16", out="bfloat16", tail="bfloat16", l2norm="hf"),
             name="decode_b233"),
        # three drafted tokens and the sampled one, checked for 24 requests at once
        dict(_case("verify", batch=24, length=4, state="bfloat16"), name="verify_b24x4"),
        # the small model in float32: launches and the chunk chain of one short sequence
        dict(_case("prefill", dtype="float32", heads=SMALL, batch=1, length=2048), name="prefill_small_fp32"),
        # one long document
        dict(_case("prefill", batch=1, length=32768), name="prefill_32768"),
        # 256-wide heads, a prompt of no round length
        dict(_case("prefill", heads=K256, batch=1, length=4099), name="prefill_k256_4099"),
        # a single chat prompt entering the layer
        dict(_case("layer", seqs=1, tokens=777, state="bfloat16", out="bfloat16", **served), name="layer_1x777"),
        # a serving engine's prefill batch: prompts of a few tokens to a few thousand, some continued
        dict(_case("layer", seqs=24, tokens=19001, state="bfloat16", out="bfloat16", **served),
             name="layer_24seq_19001"),
        # a training batch
        dict(_case("train", batch=4, length=2048), name="train_4x2048"),
        # long-context training
        dict(_case("train", batch=1, length=32768), name="train_1x32768"),
        # packed training documents of uneven lengths
        dict(_case("train", seqs=7, tokens=6011), name="train_packed_7seq"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed kinds' ranges, none dearer than the dearest listed."""
    kind = rng.choice(["decode", "verify", "prefill", "layer", "train"])
    sixteen = rng.choice(["bfloat16", "bfloat16", "float16"])
    if kind == "decode":
        return _case(kind, batch=_log_int(rng, 1, 256), state=rng.choice(["float32", "bfloat16"]),
                     tail=rng.choice(["float32", "bfloat16"]), out=rng.choice(["float32", "bfloat16"]),
                     l2norm=rng.choice(["max", "hf"]))
    if kind == "verify":
        return _case(kind, dtype=sixteen, batch=_log_int(rng, 1, 64), length=rng.randint(2, 4),
                     state=rng.choice(["float32", "bfloat16"]))
    if kind == "layer":
        tokens = _log_int(rng, 64, 32768)
        return _case(kind, seqs=_log_int(rng, 1, min(64, tokens // 8)), tokens=tokens,
                     state=rng.choice(["float32", "bfloat16"]), tail=rng.choice(["float32", "bfloat16"]),
                     out=rng.choice(["float32", "bfloat16"]), l2norm=rng.choice(["max", "hf"]))
    top = 32768
    shape = rng.choice(["wide", "wide", "wide", "small"] + (["k256"] if kind == "prefill" else []))
    dtype, heads = sixteen, WIDE
    if shape == "small":
        dtype, heads = "float32", SMALL
    elif shape == "k256":
        heads, top = K256, 12288
    tokens = _log_int(rng, 65, top)
    many = _log_int(rng, 1, min(16, max(1, tokens // 16)))
    if many > 1 and rng.random() < 0.5:
        return _case(kind, dtype=dtype, heads=heads, seqs=many, tokens=tokens)
    return _case(kind, dtype=dtype, heads=heads, batch=many, length=max(5, tokens // many))


def _lengths(case):
    """Uneven lengths of the packed sequences, the same for every seed."""
    seqs, tokens = case["seqs"], case["tokens"]
    rng = random.Random(seqs * 1000003 + tokens)
    share = [math.exp(rng.gauss(0.0, 1.0)) for _ in range(seqs)]
    lengths = [1 + int((tokens - seqs) * s / sum(share)) for s in share]
    lengths[-1] += tokens - sum(lengths)
    return lengths


def _sizes(case):
    """(batch, length, sequences) of the operator's call."""
    if "seqs" in case:
        return 1, case["tokens"], case["seqs"]
    return case["batch"], case["length"], case["batch"]


def _channels(case):
    return 2 * case["hk"] * case["dk"] + case["hv"] * case["dv"]


def _width(case):
    return _channels(case) + case["hv"] * case["dv"] + 2 * case["hv"]


class _Maker:
    """Inputs on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(*shape, device="cuda", generator=self.gen)

    def uniform(self, *shape):
        return torch.rand(*shape, device="cuda", generator=self.gen)

    def order(self, n):
        return torch.randperm(n, device="cuda", generator=self.gen)

    def layer(self, case):
        """conv weight, A_log, dt_bias, o_norm of a layer."""
        weight = (self.uniform(_channels(case), CONV) * 2 - 1) / CONV ** 0.5
        a_log = (self.uniform(case["hv"]) * 15.9 + 0.1).log()
        return weight, a_log, self.normal(case["hv"]) - 4, self.uniform(case["dv"]) + 0.5

    def tails(self, case, slots):
        """A pool of conv tails in a serving cache's channel-major layout."""
        return self.normal(slots, _channels(case), CONV - 1).to(DTYPES[case["tail"]]).transpose(1, 2)

    def states(self, case, slots):
        return (self.normal(slots, case["hv"], case["dk"], case["dv"]) * 0.05).to(DTYPES[case["state"]])

    def operands(self, case, batch, length):
        """q, k (unit length), v, g, beta as a layer hands them to the operator."""
        dtype = DTYPES[case["dtype"]]
        q = F.normalize(self.normal(batch, length, case["hk"], case["dk"]), dim=-1).to(dtype)
        k = F.normalize(self.normal(batch, length, case["hk"], case["dk"]), dim=-1).to(dtype)
        v = self.normal(batch, length, case["hv"], case["dv"]).to(dtype)
        _, a_log, dt_bias, _ = self.layer(case)
        g = -a_log.exp() * F.softplus(self.normal(batch, length, case["hv"]) + dt_bias)
        beta = torch.sigmoid(self.normal(batch, length, case["hv"]))
        return q, k, v, g, beta


def prepare(case, seed):
    make = _Maker(seed)
    kind = case["kind"]
    if kind == "decode":
        batch = case["batch"]
        slots = batch + batch // 8 + 1
        weight, a_log, dt_bias, o_norm = make.layer(case)
        return dict(case=case, z=make.normal(batch, _width(case)).to(DTYPES[case["dtype"]]),
                    tails=make.tails(case, slots), weight=weight, a_log=a_log, dt_bias=dt_bias, o_norm=o_norm,
                    states=make.states(case, slots), slots=make.order(slots)[:batch].to(torch.int32))
    if kind == "verify":
        batch, length = case["batch"], case["length"]
        order = make.order(batch * (length + 1)).to(torch.int32)
        q, k, v, g, beta = make.operands(case, batch, length)
        return dict(case=case, q=q, k=k, v=v, g=g, beta=beta, states=make.states(case, batch * (length + 1)),
                    slots=order[:batch].contiguous(), token_slots=order[batch:].view(batch, length).contiguous())
    batch, length, nseq = _sizes(case)
    cu = None
    if "seqs" in case:
        bounds = [0]
        for n in _lengths(case):
            bounds.append(bounds[-1] + n)
        cu = torch.tensor(bounds, dtype=torch.int32, device="cuda")
    if kind == "layer":
        slots = nseq + nseq // 8 + 1
        weight, a_log, dt_bias, o_norm = make.layer(case)
        # two in three requests are new, the others continue a prompt taken in pieces
        return dict(case=case, z=make.normal(length, _width(case)).to(DTYPES[case["dtype"]]), cu=cu,
                    tails=make.tails(case, slots), weight=weight, a_log=a_log, dt_bias=dt_bias, o_norm=o_norm,
                    states=make.states(case, slots), slots=make.order(slots)[:nseq].to(torch.int32),
                    started=make.uniform(nseq) < 1 / 3)
    q, k, v, g, beta = make.operands(case, batch, length)
    h0 = make.normal(nseq, case["hv"], case["dk"], case["dv"]) * 0.02
    state = dict(case=case, q=q, k=k, v=v, g=g, beta=beta, h0=h0, cu=cu)
    if kind == "train":
        for name in ("q", "k", "v", "g", "beta", "h0"):
            state[name].requires_grad_(True)
        state["grad_o"] = make.normal(batch, length, case["hv"], case["dv"]) * 0.1
        state["grad_h"] = make.normal(nseq, case["hv"], case["dk"], case["dv"]) * 0.1
    return state


def run(state):
    case, s = state["case"], state
    hk, hv, dk, dv = case["hk"], case["hv"], case["dk"], case["dv"]
    kind = case["kind"]
    if kind == "decode":
        hs = decode_layer_step(s["z"], s["tails"], s["weight"], s["a_log"], s["dt_bias"], s["states"], s["o_norm"],
                               hk, dk, hv, dv, s["slots"], case["l2norm"], EPS, out_dtype=DTYPES[case["out"]])
        return {"hs": hs, "states": s["states"], "tails": s["tails"]}
    if kind == "verify":
        o, states = recurrent_fwd(s["q"], s["k"], s["v"], s["g"], s["beta"], dk ** -0.5, s["states"], s["states"],
                                  s["slots"], out_dtype=DTYPES[case["dtype"]], token_state_idx=s["token_slots"])
        return {"o": o, "states": states}
    if kind == "layer":
        q, k, v, g, beta, gate = layer_prologue_varlen(
            s["z"], s["cu"], s["tails"], s["weight"], s["a_log"], s["dt_bias"], hk, dk, hv, dv, s["slots"],
            s["started"], case["l2norm"])
        hs = chunk_layer_fwd_slots(q, k, v, g, beta, dk ** -0.5, s["states"], s["slots"], gate, s["o_norm"], EPS,
                                   s["cu"], s["started"], out_dtype=DTYPES[case["out"]])
        return {"hs": hs, "states": s["states"], "tails": s["tails"]}
    if kind == "prefill":
        o, final = gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], dk ** -0.5, s["h0"], "hip", s["cu"])
        return {"o": o, "final": final}
    inputs = [s[name] for name in ("q", "k", "v", "g", "beta", "h0")]
    o, final = gated_delta_rule(*inputs[:5], dk ** -0.5, inputs[5], "hip", s["cu"])
    grads = torch.autograd.grad([o, final], inputs, [s["grad_o"], s["grad_h"]])
    return {"o": o.detach(), "final": final.detach(), "grads": list(grads)}


def work(case):
    hk, hv, dk, dv = case["hk"], case["hv"], case["dk"], case["dv"]
    size = {name: 4 if case.get(name) == "float32" else 2 for name in ("dtype", "state", "tail", "out")}
    kind = case["kind"]
    if kind in ("decode", "verify"):
        batch, length = case["batch"], case.get("length", 1)
        state = batch * hv * dk * dv * size["state"]
        flops = batch * length * hv * 7 * dk * dv
        if kind == "verify":  # the state read, and written after every token
            tensors = batch * length * ((2 * hk * dk + 2 * hv * dv) * size["dtype"] + 8 * hv)
            return {"bytes": state * (1 + length) + tensors, "flops": flops}
        tails = 2 * batch * (CONV - 1) * _channels(case) * size["tail"]
        rows = batch * (_width(case) * size["dtype"] + hv * dv * size["out"])
        return {"bytes": 2 * state + tails + rows + 4 * CONV * _channels(case), "flops": flops}
    batch, length, nseq = _sizes(case)
    tokens = batch * length
    # the chunked algorithm's products (64-token chunks), as bench.py counts them
    forward = tokens * hv * (2 * CHUNK * (3 * dk + 2 * dv) + 6 * dk * dv + 2 * CHUNK * CHUNK / 3)
    states = nseq * hv * dk * dv
    if kind == "layer":
        tails = 2 * nseq * (CONV - 1) * _channels(case) * size["tail"]
        rows = tokens * (_width(case) * size["dtype"] + hv * dv * size["out"])
        return {"bytes": rows + tails + 2 * states * size["state"], "flops": forward}
    qkv = tokens * (2 * hk * dk + hv * dv) * size["dtype"]
    gates = tokens * hv * 8
    if kind == "prefill":
        return {"bytes": qkv + gates + tokens * hv * dv * 4 + 8 * states, "flops": forward}
    backward = tokens * hv * (18 * dk * dv + 10 * CHUNK * dv + 12 * CHUNK * dk + 14 * CHUNK * CHUNK / 3)
    # both directions read the operands; o, its gradient and the gradients of every operand pass once
    return {"bytes": 2 * (qkv + gates) + 2 * tokens * hv * dv * 4 + qkv + gates + 5 * 4 * states,
            "flops": forward + backward}


def tolerance(case):
    """About four times what the path is off from its 64-bit value: with 16-bit
    operands and outputs 1.1e-3 to 3.4e-3 (the outputs' own rounding, and the
    rounded q, k, v between the layer's calls); with float32 ones 2e-4 to
    4.6e-4 (the chunk algorithm's products of 16-bit parts)."""
    return {"rel": 1e-2 if case["dtype"] != "float32" else 2e-3}


# ----------------------------------------------------------------------------
# The same results in 64 bits, in plain torch.
# ----------------------------------------------------------------------------
def _heads(x, hv):
    return x.repeat_interleave(hv // x.shape[2], dim=2)


def _tokenwise(q, k, v, g, beta, scale, state):
    """Token by token: o [B,T,H,V] and the state after every token [B,T,H,K,V]."""
    rows, states = [], []
    for t in range(q.shape[1]):
        state = state * g[:, t, :, None, None].exp()
        u = (v[:, t] - (state * k[:, t, :, :, None]).sum(2)) * beta[:, t, :, None]
        state = state + k[:, t, :, :, None] * u[:, :, None, :]
        rows.append((state * q[:, t, :, :, None]).sum(2) * scale)
        states.append(state)
    return torch.stack(rows, 1), torch.stack(states, 1)


def _chunkwise(q, k, v, g, beta, scale, state):
    """The recurrence by chunks of CHUNK tokens; q, k, v [B,T,H,*], g and beta
    [B,T,H], state [B,H,K,V]; (o [B,T,H,V], the final state)."""
    batch, length, heads = g.shape
    n = -(-length // CHUNK)

    def chunks(x):  # [B,T,H,*] -> [n,B,H,C,*]; padded tokens leave the state alone
        x = F.pad(x, [0, 0] * (x.ndim - 2) + [0, n * CHUNK - length])
        return x.reshape(batch, n, CHUNK, heads, -1).permute(1, 0, 3, 2, 4)

    q, k, v, beta = chunks(q * scale), chunks(k), chunks(v), chunks(beta[..., None])
    c = chunks(g[..., None]).cumsum(-2)
    lower = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device).tril()
    decay = (c - c.transpose(-1, -2)).masked_fill(~lower, -math.inf).exp()
    power = -(beta * (k @ k.transpose(-1, -2)) * decay).tril(-1)
    eye = torch.eye(CHUNK, dtype=q.dtype, device=q.device)
    inverse = eye + power
    for _ in range(5):  # (I + A)^-1 = (I - A)(I + A^2)(I + A^4) ..., A^64 = 0
        power = power @ power
        inverse = inverse @ (eye + power)
    inverse = inverse * beta.transpose(-1, -2)
    among = (q @ k.transpose(-1, -2)) * decay
    gamma, last = c.exp(), c[..., -1:, :]
    k_in, q_in, k_out, end = k * gamma, q * gamma, k * (last - c).exp(), last.exp()
    rows = []
    for i in range(n):
        u = inverse[i] @ (v[i] - k_in[i] @ state)
        rows.append(q_in[i] @ state + among[i] @ u)
        state = state * end[i] + k_out[i].transpose(-1, -2) @ u
    o = torch.stack(rows).permute(1, 0, 3, 2, 4).reshape(batch, n * CHUNK, heads, -1)
    return o[:, :length], state


def _convolve(rows, tail, weight):
    """SiLU of the causal depthwise convolution of tail ++ rows ([T,C] each), and the new tail."""
    full = torch.cat((tail, rows))
    y = sum(full[j:j + rows.shape[0]] * weight[:, j] for j in range(CONV))
    return F.silu(y), full[full.shape[0] - (CONV - 1):]


def _layer_operands(case, rows, tail, s):
    """q, k, v, g, beta [1,T,H,*] (q and k repeated), gate [T,Hv,V], new tail of one sequence's projection rows."""
    hk, hv, dk, dv = case["hk"], case["hv"], case["dk"], case["dv"]
    channels, length = _channels(case), rows.shape[0]
    y, tail = _convolve(rows[:, :channels], tail, s["weight"].double())
    gate, a, b = rows[:, channels:].split((hv * dv, hv, hv), dim=-1)
    qk = y[:, :2 * hk * dk].reshape(1, length, 2 * hk, dk)
    if case["l2norm"] == "max":
        qk = F.normalize(qk, dim=-1, eps=1e-6)
    else:
        qk = qk * (qk.square().sum(-1, keepdim=True) + 1e-6).rsqrt()
    q, k = _heads(qk[:, :, :hk], hv), _heads(qk[:, :, hk:], hv)
    g = -s["a_log"].double().exp() * F.softplus(a + s["dt_bias"].double())
    return (q, k, y[:, 2 * hk * dk:].reshape(1, length, hv, dv), g[None], torch.sigmoid(b)[None],
            gate.reshape(length, hv, dv), tail)


def _epilogue(o, gate, o_norm):
    o = o * (o.square().mean(-1, keepdim=True) + EPS).rsqrt()
    return (o * o_norm.double() * F.silu(gate)).flatten(-2)


def _exact_layer(case, s):
    """decode (each row of z a sequence of its own) and layer (rows packed by cu)."""
    z, states, tails = s["z"].double(), s["states"].double(), s["tails"].double()
    slots = s["slots"].tolist()
    bounds = list(range(len(slots) + 1)) if s.get("cu") is None else s["cu"].tolist()
    started = [True] * len(slots) if s.get("started") is None else s["started"].tolist()
    hs = []
    for n, slot in enumerate(slots):
        tail, state = tails[slot], states[slot:slot + 1]
        if not started[n]:
            tail, state = torch.zeros_like(tail), torch.zeros_like(state)
        if s.get("cu") is not None:  # the tail joins the inputs in their dtype
            tail = tail.to(DTYPES[case["dtype"]]).double()
        q, k, v, g, beta, gate, tail = _layer_operands(case, z[bounds[n]:bounds[n + 1]], tail, s)
        o, state = _chunkwise(q, k, v, g, beta, case["dk"] ** -0.5, state)
        hs.append(_epilogue(o[0], gate, s["o_norm"]))
        tails[slot], states[slot] = tail, state[0]
    return {"hs": torch.cat(hs), "states": states, "tails": tails}


def exact(case, seed):
    s = prepare(case, seed)
    kind, hv, scale = case["kind"], case["hv"], case["dk"] ** -0.5
    if kind in ("decode", "layer"):
        out = _exact_layer(case, s)
        if kind == "layer":
            out["hs"] = out["hs"][None]
        return out
    names = ("q", "k", "v", "g", "beta")
    if kind == "verify":
        q, k, v, g, beta = (s[name].double() for name in names)
        states = s["states"].double()
        o, after = _tokenwise(_heads(q, hv), _heads(k, hv), v, g, beta, scale, states[s["slots"].long()])
        states[s["token_slots"].long().flatten()] = after.flatten(0, 1)
        return {"o": o, "states": states}
    train = kind == "train"
    inputs = [s[name].detach().double().requires_grad_(train) for name in names + ("h0",)]
    with torch.set_grad_enabled(train):
        q, k, v, g, beta, h0 = inputs
        q, k = _heads(q, hv), _heads(k, hv)
        if s["cu"] is None:
            o, final = _chunkwise(q, k, v, g, beta, scale, h0)
        else:
            bounds, parts = s["cu"].tolist(), []
            for n, (lo, hi) in enumerate(zip(bounds, bounds[1:])):
                parts.append(_chunkwise(*(x[:, lo:hi] for x in (q, k, v, g, beta)), scale, h0[n:n + 1]))
            o, final = torch.cat([p[0] for p in parts], 1), torch.cat([p[1] for p in parts])
        if not train:
            return {"o": o, "final": final}
        grads = torch.autograd.grad([o, final], inputs, [s["grad_o"].double(), s["grad_h"].double()])
    return {"o": o.detach(), "final": final.detach(), "grads": list(grads)}
