"""The work that serving a mixture-of-experts model puts on this framework.

A pass is what one model step asks of the expert layers: decode steps of a few
tokens through a stack of layers (each with its own weights, so that nothing
of a layer is left in the caches when its turn comes again), batches of some
dozens of running sequences, and prefill chunks of up to thousands of tokens,
in the three weight formats, fp16 and bf16, from router output or from router
logits.  Shapes are those of the repository's configurations and benchmark:
H=2048 I=768 E=128 top-8, H=3072 I=1536 E=256 top-8 and H=2048 I=512 E=128
top-10, and generic ones around them.
"""
from __future__ import annotations

import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "moe-ascend-opt_amd"))

import nanovllm_moe  # noqa: E402
from nanovllm_moe import formats as fmt  # noqa: E402
from nanovllm_moe.synthetic import zipf_routing  # noqa: E402

GROUP = 128
QUANT = {"q8_0": 0, "q4_0": 1, "w4a16": 2}
DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, quant, E, H, I, K, T, layers=1, act="bf16", scales=None, routing="uniform", call="op"):
    """call: "op" = moe_forward, "graph" = moe_forward_out of every layer captured once
    and replayed, "logits" = moe_forward_logits (router top-k and softmax included)."""
    c = {"quant": quant, "E": E, "H": H, "I": I, "top_k": K, "tokens": T, "layers": layers, "act": act,
         "scales": scales or ("bf16" if quant == "w4a16" else "fp16"), "routing": routing, "call": call}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one user's decode step, replayed from a graph: the latency of every generated token
        _case("w4a16_decode_1", "w4a16", 128, 2048, 768, 8, 1, layers=8, call="graph"),
        # a small batch of users
        _case("w4a16_decode_8", "w4a16", 128, 2048, 768, 8, 8, layers=4, call="graph"),
        # continuous batching: an odd number of running sequences, fp16 model, straight from the router logits
        _case("w4a16_batch_37_fp16", "w4a16", 128, 2048, 768, 8, 37, layers=3, act="fp16", scales="fp16",
              call="logits"),
        # a wide layer with many experts at the batch size of a busy server
        _case("w4a16_wide_64", "w4a16", 256, 3072, 1536, 8, 64),
        # skewed expert popularity: a few hot experts, many nearly idle ones
        _case("w4a16_zipf_512", "w4a16", 128, 2048, 768, 8, 512, routing="zipf"),
        # a whole prompt or a full prefill chunk
        _case("w4a16_prefill_4096", "w4a16", 128, 2048, 768, 8, 4096),
        # the wide layer's prefill chunk, an odd number of tokens: about 40 rows an expert
        _case("w4a16_wide_1333", "w4a16", 256, 3072, 1536, 8, 1333),
        # decode with 8-bit weights, a few sequences (speculative tokens or a small batch)
        _case("q8_0_decode_3", "q8_0", 128, 2048, 768, 8, 3, layers=4, call="graph"),
        # 8-bit weights, an odd prompt length
        _case("q8_0_prefill_1021", "q8_0", 128, 2048, 768, 8, 1021),
        # top-10 layer, eager calls as the op's Python caller makes them
        _case("q4_0_top10_decode_7", "q4_0", 128, 2048, 512, 10, 7, layers=6),
        # continuous batching with 4-bit weights
        _case("q4_0_batch_45", "q4_0", 128, 2048, 768, 8, 45, layers=3),
        # a full prefill chunk with 4-bit weights
        _case("q4_0_prefill_4096", "q4_0", 128, 2048, 768, 8, 4096),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    quant = rng.choice(["w4a16", "w4a16", "q8_0", "q4_0"])
    E, H, I, K = rng.choice([(128, 2048, 768, 8), (128, 2048, 768, 8), (256, 3072, 1536, 8), (128, 2048, 512, 10),
                             (64, 2048, 1024, rng.randint(4, 8)), (32, 4096, 768, rng.randint(1, 6)),
                             (rng.randint(17, 200), 512 * rng.randint(2, 6), 128 * rng.randint(2, 10),
                              rng.randint(1, 12))])
    T = log_int(1, 4096)
    while T * K * H * I > 4096 * 8 * 2048 * 768:   # no more work than the largest listed case
        T = max(1, T // 2 - rng.randint(0, 1))
    call = rng.choice(["graph", "op", "logits"]) if T <= 64 else rng.choice(["op", "op", "logits"])
    act = rng.choice(["bf16", "bf16", "fp16"])
    scales = rng.choice(["bf16", "fp16"])
    routing = "uniform" if call == "logits" else rng.choice(["uniform", "uniform", "zipf"])
    layers = min(rng.randint(2, 4) if T <= 64 else 1, max(1, 256 * 3072 * 1536 // (E * H * I)))
    return _case(None, quant, E, H, I, K, T, layers=layers, act=act, scales=scales,
                 routing=routing, call=call)


def _gen(seed, layer, what):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 131 + layer) * 17 + what)


def _weights(c, seed, layer):
    """The wire tensors of a layer: N(0, 0.02) weights quantized in the layer's format."""
    E, H, I = c["E"], c["H"], c["I"]
    sdt = DTYPE[c["scales"]]
    out = []
    for what, (N, K) in enumerate(((2 * I, H), (H, I))):
        g = _gen(seed, layer, what)
        parts = []
        step = max(1, (1 << 26) // (N * K))   # experts at a time
        for e in range(0, E, step):
            w = torch.randn(min(step, E - e), N, K, generator=g, device="cuda") * 0.02
            if c["quant"] == "w4a16":
                parts.append(fmt.awq_quantize(w, GROUP, sdt))
            elif c["quant"] == "q4_0":
                parts.append(fmt.q4_0_quantize(w, sdt))
            else:
                b = w.reshape(w.shape[0], N, K // 32, 32)
                d = (b.abs().amax(-1) / 127.0).to(sdt)
                q = torch.round(b / d.float().unsqueeze(-1)).clamp_(-127, 127).to(torch.int8)
                parts.append((q.reshape(w.shape), d))
        out += [torch.cat(p) for p in zip(*parts)]
    return out


def _inputs(c, seed, layer):
    """Hidden states, router logits, and the router's picks."""
    T, E, K = c["tokens"], c["E"], c["top_k"]
    g = _gen(seed, layer, 2)
    x = torch.randn(T, c["H"], generator=g, device="cuda").to(DTYPE[c["act"]])
    logits = torch.randn(T, E, generator=g, device="cuda")
    if c["routing"] == "zipf":
        ids, w = zipf_routing(T, E, K, seed=(int(seed) * 131 + layer) % (1 << 31))
        ids, w = ids.cuda(), w.cuda()
    else:
        val, ids = torch.topk(logits, K, dim=-1)
        ids, w = ids.to(torch.int32), torch.softmax(val, dim=-1)
    return x, logits, ids.contiguous(), w.contiguous()


def prepare(case, seed):
    nanovllm_moe.load()
    c = case
    layers = []
    for n in range(c["layers"]):
        h = torch.classes.nanovllm.MoEInfer(c["E"], c["H"], c["I"], QUANT[c["quant"]])
        wire = _weights(c, seed, n)
        if c["quant"] == "w4a16":
            h.store_awq_repack(*wire, GROUP)
        else:
            h.store_quantized_repack(*wire)
        del wire
        layers.append((h, *_inputs(c, seed, n)))
    graph, outs = None, None
    if c["call"] == "graph":
        outs = [torch.empty_like(x) for _, x, _, _, _ in layers]
        for (h, x, _, ids, w), y in zip(layers, outs):   # the first call sizes the workspace
            torch.ops.nanovllm.moe_forward_out(x, ids, w, h, y)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for (h, x, _, ids, w), y in zip(layers, outs):
                torch.ops.nanovllm.moe_forward_out(x, ids, w, h, y)
    return {"graph": graph, "outs": outs, "layers": layers, "call": c["call"], "top_k": c["top_k"]}


def run(state):
    if state["call"] == "graph":
        state["graph"].replay()
        return state["outs"]
    if state["call"] == "logits":
        return [torch.ops.nanovllm.moe_forward_logits(x, logits, state["top_k"], True, h)
                for h, x, logits, _, _ in state["layers"]]
    return [torch.ops.nanovllm.moe_forward(x, ids, w, h) for h, x, _, ids, w in state["layers"]]


def work(case):
    """The routed experts' weights once, the hidden states in and out, the routing; the products of every pair."""
    c = case
    T, K, H, E = c["tokens"], c["top_k"], c["H"], c["E"]
    if c["routing"] == "zipf":
        used = len(np.unique(zipf_routing(T, E, K, seed=0)[0].numpy()))
    else:
        used = E * (1.0 - (1.0 - K / E) ** T)
    per = used * fmt.bytes_per_expert(QUANT[c["quant"]], H, c["I"], GROUP) + 4 * T * H
    per += 4 * T * E if c["call"] == "logits" else 8 * T * K
    return {"bytes": c["layers"] * per, "flops": c["layers"] * 6.0 * T * K * H * c["I"]}


def tolerance(case):
    # About four times the distance from 64 bits: it is that of one rounding of the intermediate (W4A16) and
    # of the result to 16 bits.  Q8_0 / Q4_0: of the result alone, plus the intermediates that lie between two
    # 8-bit codes.
    bits = 8.0 if case["act"] == "bf16" else 1.0
    if case["quant"] == "w4a16":
        return {"rel": 1.4e-3 * bits, "max": 1e-2 * bits}
    return {"rel": 1.2e-3 * bits, "max": 1e-2 * bits}


def _q8(v):
    """Q8_0 along the last dimension, as the formats define it, in the precision of v: the values it stands for."""
    b = v.reshape(*v.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    q = torch.round(b * torch.where(d == 0, 0.0, 1.0 / d))
    return (q.clamp(-127, 127) * d).reshape(v.shape)


def exact(case, seed):
    c = case
    out = []
    for n in range(c["layers"]):
        wire = _weights(c, seed, n)
        x, _, ids, w = _inputs(c, seed, n)
        val = w.double()
        x = x.double() if c["quant"] == "w4a16" else _q8(x.float()).double()
        y = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
        for e in torch.unique(ids).tolist():
            t, k = torch.nonzero(ids == e, as_tuple=True)
            w1, w2 = (_dequant(c, wire, p, e) for p in (0, 1))
            gu = x[t] @ w1.t()
            h = torch.nn.functional.silu(gu[:, :c["I"]]) * gu[:, c["I"]:]
            if c["quant"] != "w4a16":
                h = _q8(h)
            y.index_add_(0, t, (h @ w2.t()) * val[t, k].unsqueeze(1))
        out.append(y)
    return out


def _dequant(c, wire, p, e):
    """Projection p (0 gate and up, 1 down) of expert e in 64 bits, [N, K]."""
    if c["quant"] == "w4a16":
        q, z, s = (t[e].to(torch.int64) & 0xFFFFFFFF if t.dtype == torch.int32 else t[e].double()
                   for t in wire[3 * p:3 * p + 3])
        shift = torch.tensor([0, 16, 4, 20, 8, 24, 12, 28], device=q.device)   # column n of 8: its nibble
        q, z = (((t.unsqueeze(-1) >> shift) & 15).reshape(t.shape[0], -1).double() for t in (q, z))
        return ((q - z.repeat_interleave(GROUP, 0)) * s.repeat_interleave(GROUP, 0)).t()
    q, d = wire[2 * p][e], wire[2 * p + 1][e].double()
    if c["quant"] == "q4_0":
        q = (q.to(torch.int64).unsqueeze(-1) >> torch.arange(0, 32, 4, device=q.device)) & 15
        q = q.reshape(q.shape[0], -1) - 8
    return q.double() * d.repeat_interleave(32, 1)
