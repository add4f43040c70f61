"""Timed cases of the MoE path: what a decoder that runs on this package has it do.

Three kinds of call:

  layer    MoeBlock.forward, one layer or a chain of layers (out = x + MoE(RMSNorm(x)))
  experts  FusedExperts.forward, the op layer (mul_mv_id / mul_mm_id, silu_mul, combine)
           for callers that route themselves
  mul_mv   ops.mul_mv, the plain quantised mat-vec (the lm_head, dense projections)

Weights are random quants whose scales make them centred with a standard
deviation near 1/sqrt(k), as trained matrices are; activations are normal with
log-normal channel gains (a few channels far larger than the rest); routers and
selection biases are normal.  Everything is made on the GPU from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from maxuna_amd import ops
from maxuna_amd.gguf import ExpertStack, GgmlDType, row_bytes
from maxuna_amd.moe import FusedExperts, MoeBlock, MoeConfig, SharedExpert

RMS_EPS = 1e-6
WEIGHTS_SUM_FLOOR = 6.103515625e-5
# (value range of the quants, their root mean square about the centre, root mean square of the sub-block scale)
QUANT = {"Q4_K": (15, 4.61, 36.4), "Q5_K": (31, 9.23, 36.4), "Q6_K": (63, 18.5, 73.9), "Q8_0": (255, 73.9, 1.0)}


def _layer(name, hidden, ff, experts, top_k, gate, down, shared, t, layers=1, rms=False, bias=0.1, scale=1.0):
    return dict(name=name, kind="layer", hidden=hidden, ff=ff, experts=experts, top_k=top_k, gate=gate, down=down,
                shared=shared, t=t, layers=layers, rms=rms, bias=bias, scale=scale)


def listed():
    return [
        # one token through the smallest layer: launches and latency only
        _layer("small_layer_t1", 1024, 512, 64, 4, "Q4_K", "Q4_K", False, 1, bias=0.0),
        # batch-1 decode, four consecutive decoder layers' FFN halves at the benchmark's width
        _layer("decode_chain4_t1", 4096, 1536, 256, 10, "Q4_K", "Q6_K", True, 1, layers=4, rms=True),
        # the same at the Laguna width (hidden 3072, ff 1024, scale 2.5)
        _layer("decode_laguna_chain4_t1", 3072, 1024, 256, 10, "Q4_K", "Q6_K", True, 1, layers=4, rms=True, scale=2.5),
        # a few concurrent sequences, higher-precision quants
        _layer("decode_q5k_t4", 5120, 1536, 128, 8, "Q5_K", "Q6_K", True, 4),
        # an odd small batch over few large 8-bit experts
        _layer("decode_q8_t9", 3072, 2048, 64, 4, "Q8_0", "Q8_0", False, 9),
        # speculative verification of 16 tokens
        _layer("verify_t16", 4096, 1536, 256, 10, "Q4_K", "Q6_K", True, 16),
        # a short prompt or a large decode batch at a wide model
        _layer("batch_wide_t100", 7168, 2048, 256, 8, "Q4_K", "Q5_K", False, 100),
        # prompts: a ragged chunk at the Laguna width, and the benchmark's 2048 tokens with skewed routing
        _layer("prefill_laguna_t925", 3072, 1024, 256, 10, "Q4_K", "Q6_K", True, 925, rms=True, scale=2.5),
        _layer("prefill_t2048", 4096, 1536, 256, 10, "Q4_K", "Q6_K", True, 2048, bias=0.5),
        # the op layer at a prompt of 512 tokens
        dict(name="experts_t512", kind="experts", hidden=4096, ff=1536, experts=256, top_k=10, gate="Q4_K",
             down="Q6_K", t=512),
        # the vocabulary projection: of one decoded token, and of all tokens of a verified block
        dict(name="lm_head_t1", kind="mul_mv", n_out=100352, k=3072, dtype="Q6_K", t=1),
        dict(name="lm_head_t16", kind="mul_mv", n_out=100352, k=3072, dtype="Q6_K", t=16),
    ]


def _spread(rng, lo, hi):
    """A whole number of lo..hi, even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# gate/up and down types that go together in published files
MIXES = [("Q4_K", "Q6_K"), ("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q4_K", "Q5_K"), ("Q5_K", "Q6_K"), ("Q5_K", "Q5_K"),
         ("Q6_K", "Q4_K"), ("Q6_K", "Q6_K"), ("Q8_0", "Q8_0")]
# (hidden, ff, experts, top_k, shared): the geometries of the tests and the benchmark
SHAPES = [(1024, 512, 64, 4, False), (2048, 768, 128, 8, True), (3072, 1024, 256, 10, True), (3072, 2048, 64, 4, False),
          (4096, 1536, 256, 10, True), (5120, 1536, 128, 8, True), (6144, 2816, 64, 4, True), (7168, 2048, 256, 8, False)]


def draw(rng):
    cap = 0.4 * work(listed()[8])["flops"]
    while True:
        kind = rng.choice(["layer"] * 5 + ["experts", "mul_mv"])
        if kind == "mul_mv":
            case = dict(kind=kind, n_out=_spread(rng, 1000, 100352), k=256 * _spread(rng, 4, 24),
                        dtype=rng.choice(sorted(QUANT)), t=_spread(rng, 1, 24))
        else:
            gate, down = rng.choice(MIXES)
            hidden, ff, experts, top_k, shared = rng.choice(SHAPES)
            if rng.random() < 0.4:  # other widths, expert counts and top-k
                step = 32 if gate == down == "Q8_0" else 256
                hidden = step * _spread(rng, 1024 // step, 7168 // step)
                ff = step * _spread(rng, 512 // step, 2816 // step)
                experts = _spread(rng, 24, 256)
                top_k = rng.randint(2, 10)
            case = dict(kind=kind, hidden=hidden, ff=ff, experts=experts, top_k=top_k, gate=gate, down=down)
            if kind == "layer":
                case.update(shared=shared, t=_spread(rng, 1, 2048), layers=1, rms=rng.random() < 0.5,
                            bias=rng.choice([0.1, 0.1, 0.5]), scale=rng.choice([1.0, 2.5]))
            else:
                case.update(t=_spread(rng, 1, 1024))
            expert_bytes = 2 * ff * row_bytes(GgmlDType[gate], hidden) + hidden * row_bytes(GgmlDType[down], ff)
            if experts * expert_bytes > 8e9:
                continue
        if work(case)["flops"] <= cap:
            return case


# ---- inputs -------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _activations(g, t, dim):
    return _normal(g, t, dim) * torch.exp(0.5 * _normal(g, dim))


def _blocks(g, dtype, rows, k):
    """Raw GGUF blocks of `rows` rows of k weights."""
    name = dtype.name
    n_blocks = rows * k // dtype.block_size
    raw = torch.randint(0, 256, (n_blocks, dtype.type_size), dtype=torch.uint8, device="cuda", generator=g)
    span, q_rms, s_rms = QUANT[name]
    d = (0.5 + torch.rand(n_blocks, device="cuda", generator=g)) / (q_rms * s_rms * math.sqrt(k))
    f16 = lambda v: v.to(torch.float16).view(torch.uint8).reshape(n_blocks, 2)  # noqa: E731
    if name in ("Q4_K", "Q5_K"):
        raw[:, 0:2] = f16(d)
        # the minimum of a sub-block is span / 2 steps of its scale: sc == m and dmin = span / 2 * d
        raw[:, 2:4] = f16(d.to(torch.float16).float() * (span / 2))
        raw[:, 8:12] = raw[:, 4:8]
        raw[:, 12:16] = (raw[:, 12:16] & 15) * 17
    elif name == "Q6_K":
        raw[:, 208:210] = f16(d)
    else:
        raw[:, 0:2] = f16(d)
    return raw.reshape(-1)


def _stack(g, dtype, n_expert, n_out, k):
    dt = GgmlDType[dtype]
    return ExpertStack(_blocks(g, dt, n_expert * n_out, k), dt, n_expert, n_out, k)


def _block(g, c):
    gate, down, hidden, ff, experts = c["gate"], c["down"], c["hidden"], c["ff"], c["experts"]
    router = 0.02 * _normal(g, experts, hidden)
    bias = c["bias"] * _normal(g, experts)
    stacks = [_stack(g, gate, experts, ff, hidden), _stack(g, gate, experts, ff, hidden), _stack(g, down, experts, hidden, ff)]
    shared = None
    if c["shared"]:
        shared = SharedExpert(_stack(g, gate, 1, ff, hidden), _stack(g, gate, 1, ff, hidden), _stack(g, down, 1, hidden, ff))
    alpha = 1.0 + 0.1 * _normal(g, hidden) if c["rms"] else None
    return MoeBlock(router, bias, *stacks, MoeConfig(c["top_k"], c["scale"], True), shared=shared, rms_alpha=alpha,
                    rms_eps=RMS_EPS)


def prepare(case, seed):
    g = _generator(seed)
    if case["kind"] == "mul_mv":
        dt = GgmlDType[case["dtype"]]
        return dict(case=case, weight=_blocks(g, dt, case["n_out"], case["k"]), dtype=dt,
                    x=_activations(g, case["t"], case["k"]))
    if case["kind"] == "experts":
        t, top_k, experts = case["t"], case["top_k"], case["experts"]
        gate, down, hidden, ff = case["gate"], case["down"], case["hidden"], case["ff"]
        score = _normal(g, t, experts) + 0.5 * _normal(g, experts)
        top, ids = torch.topk(score, top_k, dim=1)
        runner = FusedExperts(_stack(g, gate, experts, ff, hidden), _stack(g, gate, experts, ff, hidden),
                              _stack(g, down, experts, hidden, ff))
        return dict(case=case, runner=runner, x=_activations(g, t, hidden), ids=ids.to(torch.int32).view(torch.uint32),
                    weights=torch.softmax(top, dim=1).contiguous())
    return dict(case=case, blocks=[_block(g, case) for _ in range(case["layers"])],
                x=_activations(g, case["t"], case["hidden"]))


def run(state):
    case = state["case"]
    if case["kind"] == "mul_mv":
        return ops.mul_mv(state["weight"], state["dtype"], case["n_out"], case["k"], state["x"])
    if case["kind"] == "experts":
        return state["runner"].forward(state["x"], state["ids"], state["weights"])
    if case["layers"] == 1:
        block, x = state["blocks"][0], state["x"]
        out, ids, w = block.forward(x, residual=x if case["rms"] else None, return_routing=True)
        return {"out": out, "ids": ids.view(torch.int32), "w": w}
    h, hidden = state["x"], []
    for block in state["blocks"]:
        h = block.forward(h, residual=h)
        hidden.append(h)
    return hidden


# ---- what a pass cannot do without --------------------------------------------------


def _touched(experts, top_k, t, spread, bias):
    """Experts that t tokens touch, on one drawn routing: the selection bias gathers tokens on few experts
    (logits of standard deviation `spread`)."""
    r = np.random.RandomState(7)
    sel = 1.0 / (1.0 + np.exp(-spread * r.standard_normal((t, experts)))) + bias * r.standard_normal(experts)
    return len(np.unique(np.argpartition(-sel, top_k - 1, axis=1)[:, :top_k]))


def work(case):
    if case["kind"] == "mul_mv":
        n_out, k, t = case["n_out"], case["k"], case["t"]
        return {"bytes": n_out * row_bytes(GgmlDType[case["dtype"]], k) + 4 * t * (k + n_out), "flops": 2 * t * n_out * k}
    hidden, ff, t, top_k, experts = case["hidden"], case["ff"], case["t"], case["top_k"], case["experts"]
    one = 2 * ff * row_bytes(GgmlDType[case["gate"]], hidden) + hidden * row_bytes(GgmlDType[case["down"]], ff)
    per_pair = 6 * hidden * ff
    if case["kind"] == "experts":
        touched = _touched(experts, top_k, t, 0.04, 0.005)
        return {"bytes": touched * one + 8 * t * (hidden + top_k), "flops": t * top_k * per_pair}
    shared = 1 if case["shared"] else 0
    spread = 0.02 * math.sqrt(hidden) * (1.0 if case["rms"] else 1.28)
    touched = _touched(experts, top_k, t, spread, case["bias"])
    nbytes = (touched + shared) * one + 4 * experts * (hidden + 1) + 8 * t * (hidden + top_k)
    flops = t * (top_k + shared) * per_pair + 2 * t * hidden * experts
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    """Below 16 tokens (32 in the op layer) and in mul_mv results are those of f32
    products and sums; from there on the expert products take f16 operands."""
    if case["kind"] == "mul_mv":
        return {"rel": 1e-6, "max": 2e-5}
    if case["t"] < (16 if case["kind"] == "layer" else 32):
        # the router's f32 logits may order near-ties in another way
        return {"rel": 2e-6, "max": 4e-5, "differ": 0.01}
    return {"rel": 2e-3, "max": 2e-2, "differ": 0.002}


# ---- the same in 64 bits ------------------------------------------------------------


def _k_scales(s):
    """Scales and minima [n, 8] of the 12 packed bytes of Q4_K / Q5_K blocks."""
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _weights(raw, dtype, rows, k):
    """[rows, k] weights in 64 bits."""
    b = raw.reshape(-1, dtype.type_size)
    n = b.shape[0]
    f16 = lambda o: b[:, o:o + 2].contiguous().view(torch.float16).double()  # noqa: E731
    name = dtype.name
    if name == "Q8_0":
        w = b[:, 2:].contiguous().view(torch.int8).double() * f16(0)
    elif name == "Q6_K":
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device).reshape(1, 1, 4, 1)
        low = torch.cat([ql & 15, ql >> 4], 2)  # parts 0..3 of a half: low nibbles of both rows, then the high ones
        q = (low | (((qh >> shift) & 3) << 4)).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = q.reshape(n, 16, 16) * sc.reshape(n, 16, 1) * f16(208).reshape(n, 1, 1)
    else:
        sc, mn = _k_scales(b[:, 4:16])
        qs = b[:, 16:144] if name == "Q4_K" else b[:, 48:176]
        qs = qs.reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if name == "Q5_K":
            bit = torch.arange(8, dtype=torch.uint8, device=b.device).reshape(1, 8, 1)
            q = q | (((b[:, 16:48].reshape(n, 1, 32) >> bit) & 1) << 4)
        w = q.double() * sc.reshape(n, 8, 1) * f16(0).reshape(n, 1, 1) - (mn * f16(2)).reshape(n, 8, 1)
    return w.reshape(rows, k)


def _expert(stack, e):
    step = stack.n_out * row_bytes(stack.dtype, stack.k)
    return _weights(stack.buffer[e * step:(e + 1) * step], stack.dtype, stack.n_out, stack.k)


def _swiglu(x, gate, up, down, e):
    g, u = x @ _expert(gate, e).T, x @ _expert(up, e).T
    return (g / (1.0 + torch.exp(-g)) * u) @ _expert(down, e).T


def _routed(x, experts, ids, w):
    out = torch.zeros_like(x)
    for e in torch.unique(ids).tolist():
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        out.index_add_(0, tok, _swiglu(x[tok], experts.gate, experts.up, experts.down, e) * w[tok, slot][:, None])
    return out


def _moe(block, h, case):
    x = h
    if case["rms"]:
        x = h / torch.sqrt((h * h).mean(1, keepdim=True) + RMS_EPS) * block.rms_alpha.double()
    probs = torch.sigmoid(x @ block.router.double().T)
    ids = torch.argsort(probs + block.exp_probs_b.double(), dim=1, descending=True, stable=True)[:, :case["top_k"]]
    w = probs.gather(1, ids)
    w = w / w.sum(1, keepdim=True).clamp_min(WEIGHTS_SUM_FLOOR) * case["scale"]
    out = _routed(x, block.experts, ids, w)
    if block.shared is not None:
        out = out + _swiglu(x, block.shared.gate, block.shared.up, block.shared.down, 0)
    return (out + h if case["rms"] else out), w


def exact(case, seed):
    state = prepare(case, seed)
    x = state["x"].double()
    if case["kind"] == "mul_mv":
        per = row_bytes(state["dtype"], case["k"])
        out = torch.empty(case["t"], case["n_out"], dtype=torch.float64, device="cuda")
        for r in range(0, case["n_out"], 8192):
            n = min(8192, case["n_out"] - r)
            out[:, r:r + n] = x @ _weights(state["weight"][r * per:(r + n) * per], state["dtype"], n, case["k"]).T
        return out
    if case["kind"] == "experts":
        return _routed(x, state["runner"], state["ids"].view(torch.int32).long(), state["weights"].double())
    if case["layers"] == 1:
        out, w = _moe(state["blocks"][0], x, case)
        return {"out": out, "ids": None, "w": w}
    hidden = []
    for block in state["blocks"]:
        x, _ = _moe(block, x, case)
        hidden.append(x)
    return hidden
