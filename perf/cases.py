"""Performance cases of the fused MoE layer: what its callers run, through the public entry points.

Kinds
  layer   fast_route_amd.layers.fused_moe.fused_moe: hidden states + router logits, bf16 (the serving entry point)
  gate    fast_route_amd.layers.stable_route.fused_moe: routing from the gate matrix, fp16 (the drop-in entry point)
  fp8     fast_route_amd.layers.fp8.fused_moe_fp8: bf16 hidden states, e4m3 weights
  route   fast_route_amd.ops: topk_softmax, then moe_align_block_size (callers that bring their own expert GEMMs)

Shapes are the ones bench.py and the tests use; token counts go from one sequence decoding to a long prefill.
"""
from __future__ import annotations

import math

import torch

from fast_route_amd.layers import fused_moe as layer_api
from fast_route_amd.layers import stable_route as gate_api
from fast_route_amd.layers.fp8 import fused_moe_fp8, prepare_weights_fp8
from fast_route_amd.ops.fused_moe import moe_align_block_size
from fast_route_amd.ops.stable_route import topk_softmax

SHAPES = {
    # 8 wide experts, near-uniform load
    "mixtral": dict(H=4096, F=14336, E=8, topk=2, zipf=False),
    "mixtral22b": dict(H=6144, F=16384, E=8, topk=2, zipf=False),
    # 64 narrow experts, Zipf-skewed load
    "fine": dict(H=2048, F=1408, E=64, topk=6, zipf=True),
    # one small layer: everything but the weight stream is launches and latency
    "small": dict(H=1024, F=3584, E=8, topk=2, zipf=False),
    # the reference's own benchmark protocol (16 experts, fp16, randn / 10)
    "protocol": dict(H=4096, F=8192, E=16, topk=2, zipf=False),
    # routing stress: 64 experts, top-6, Zipf-skewed
    "stress": dict(H=0, F=0, E=64, topk=6, zipf=True),
}


def _case(kind, shape, tokens, name=None, prepared=False, block=0):
    c = {"kind": kind, "shape": shape, "tokens": int(tokens), "prepared": bool(prepared), "block": int(block)}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one sequence decoding: two experts' weights streamed once, launch latency next to it
        _case("layer", "mixtral", 1, "mixtral_decode_1"),
        # continuous batching at decode: all experts hit by a few tokens each
        _case("layer", "mixtral", 24, "mixtral_decode_24"),
        # a small chunk of prefill, or a large decode batch: between weight streaming and compute
        _case("layer", "mixtral", 1031, "mixtral_chunk_1031"),
        # the headline batch of the layer
        _case("layer", "mixtral", 4096, "mixtral_prefill_4096"),
        # a long prefill on weights laid out once with prepare_weights
        _case("layer", "mixtral", 16384, "mixtral_prefill_16384_prepared", prepared=True),
        # many-expert models: decode batch, chunk, prefill
        _case("layer", "fine", 32, "fine_decode_32"),
        _case("layer", "fine", 509, "fine_chunk_509"),
        _case("layer", "fine", 8192, "fine_prefill_8192"),
        # quantised serving: decode and a prefill chunk
        _case("fp8", "mixtral", 16, "fp8_decode_16"),
        _case("fp8", "mixtral", 2048, "fp8_prefill_2048"),
        # the drop-in call of the reference's benchmark: gate matrix in, fp16
        _case("gate", "protocol", 700, "gate_fp16_700"),
        # routing alone on a large skewed batch
        _case("route", "stress", 65536, "route_65536", block=64),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    pick = rng.random()
    if pick < 0.30:
        return _case("layer", "mixtral", _log_uniform(rng, 1, 16384), prepared=rng.random() < 0.25)
    if pick < 0.38:
        return _case("layer", "mixtral22b", _log_uniform(rng, 1, 8192))
    if pick < 0.63:
        return _case("layer", "fine", _log_uniform(rng, 1, 8192))
    if pick < 0.70:
        return _case("layer", "small", _log_uniform(rng, 1, 4096))
    if pick < 0.83:
        return _case("fp8", "mixtral", _log_uniform(rng, 1, 8192))
    if pick < 0.93:
        return _case("gate", "protocol", _log_uniform(rng, 1, 8192))
    return _case("route", "stress", _log_uniform(rng, 256, 65536), block=rng.choice((16, 32, 64, 128)))


def _logits(gen, dev, M, E, zipf):
    noise = torch.randn(M, E, generator=gen, device=dev)
    if not zipf:
        return noise
    # log of a Zipf(1.2) law over the experts, in an order of the seed's own
    p = (torch.randperm(E, generator=gen, device=dev) + 1).double().pow(-1.2)
    return (torch.log(p / p.sum()).float()[None, :] + noise).contiguous()


def prepare(case, seed):
    s = SHAPES[case["shape"]]
    M, H, F, E, topk = case["tokens"], s["H"], s["F"], s["E"], s["topk"]
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed) & 0x7FFFFFFF)
    st = {"kind": case["kind"], "topk": topk, "E": E, "block": case["block"], "flags": 0}

    def normal(shape, dtype, std):
        return torch.empty(shape, dtype=dtype, device=dev).normal_(0.0, std, generator=gen)

    if case["kind"] == "gate":  # the reference's recipe: everything randn / 10 in fp16
        st["x"] = normal((M, H), torch.float16, 0.1)
        st["gate"] = normal((H, E), torch.float16, 0.1)
        st["w1"] = normal((E, 2 * F, H), torch.float16, 0.1)
        st["w2"] = normal((E, H, F), torch.float16, 0.1)
        return st
    st["logits"] = _logits(gen, dev, M, E, s["zipf"])
    if case["kind"] == "route":
        st["topk_weights"] = torch.empty((M, topk), dtype=torch.float32, device=dev)
        st["topk_ids"] = torch.empty((M, topk), dtype=torch.int32, device=dev)
        return st
    st["x"] = normal((M, H), torch.bfloat16, 1.0)
    w1 = normal((E, 2 * F, H), torch.bfloat16, 0.02)
    w2 = normal((E, H, F), torch.bfloat16, 0.02)
    if case["kind"] == "fp8":
        st["w1q"], st["w1s"], st["w2q"], st["w2s"] = prepare_weights_fp8(w1, w2)
        return st
    if case["prepared"]:
        w1, w2, st["flags"] = layer_api.prepare_weights(w1, w2)
    st["w1"], st["w2"] = w1, w2
    return st


def run(st):
    if st["kind"] == "layer":
        return layer_api.fused_moe(st["x"], st["w1"], st["w2"], st["logits"], st["topk"], renormalize=True,
                                   weights_prepared=st["flags"])
    if st["kind"] == "gate":
        return gate_api.fused_moe(st["x"], st["gate"], st["w1"], st["w2"], st["topk"], renormalize=True)
    if st["kind"] == "fp8":
        return fused_moe_fp8(st["x"], st["w1q"], st["w1s"], st["w2q"], st["w2s"], st["logits"], st["topk"],
                             renormalize=True)
    w, ids = topk_softmax(st["topk_weights"], st["topk_ids"], None, st["logits"], renormalize=True)
    sorted_ids, expert_ids, npost = moe_align_block_size(ids, st["block"], st["E"])
    # expert_ids is specified for the npost / block blocks in use, at least n / block of them; what lies behind is
    # memory nobody writes
    return w, ids, sorted_ids, expert_ids[: ids.numel() // st["block"]], npost


def _quantised(x):
    """Rows as e4m3 holds them (scale = largest magnitude / 448, in 32 bits), back in 64 bits."""
    scale = x.abs().amax(dim=1, keepdim=True).float() / 448.0
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    return (x.float() / scale).to(torch.float8_e4m3fn).double() * scale.double()


def exact(case, seed):
    """run()'s floating outputs in 64 bits with plain torch, from the same inputs."""
    st, topk = prepare({**case, "prepared": False}, seed), SHAPES[case["shape"]]["topk"]
    logits = (st["x"].double() @ st["gate"].double()) if case["kind"] == "gate" else st["logits"].double()
    top, ids = torch.sort(logits, dim=1, descending=True, stable=True)
    top, ids = top[:, :topk], ids[:, :topk]
    if case["kind"] == "route":
        return torch.softmax(top, dim=1), None, None, None, None
    weights, fp8 = torch.softmax(top, dim=1), case["kind"] == "fp8"
    x = _quantised(st["x"].double()) if fp8 else st["x"].double()
    out = torch.zeros_like(x)
    for e in range(st["E"]):
        token, slot = (ids == e).nonzero(as_tuple=True)
        if token.numel() == 0:
            continue
        if fp8:
            w1 = st["w1q"][e].view(torch.float8_e4m3fn).double() * st["w1s"][e].double()[:, None]
            w2 = st["w2q"][e].view(torch.float8_e4m3fn).double() * st["w2s"][e].double()[:, None]
        else:
            w1, w2 = st["w1"][e].double(), st["w2"][e].double()
        gate, up = (x[token] @ w1.t()).chunk(2, dim=1)
        act = torch.nn.functional.silu(gate) * up
        if fp8:  # the path's own formats: activated rows in bf16, quantised per row
            act = _quantised(act.bfloat16().double())
        out.index_add_(0, token, (act @ w2.t()) * weights[token, slot][:, None])
    return out


def _active_experts(M, E, topk, zipf):
    """Experts that a batch of M tokens hits, from one sample of the case's logits."""
    gen = torch.Generator(device="cpu").manual_seed(1)
    logits = _logits(gen, torch.device("cpu"), min(M, 4096), E, zipf)
    return int(torch.unique(torch.topk(logits, topk, dim=1).indices).numel())


def work(case):
    s = SHAPES[case["shape"]]
    M, H, F, E, topk = case["tokens"], s["H"], s["F"], s["E"], s["topk"]
    if case["kind"] == "route":
        n, block = M * topk, case["block"]
        # logits in; weights, ids, sorted ids (with their padding) and block table out
        return {"bytes": 4 * M * E + 8 * n + 4 * (n + E * (block - 1)) + 4 * (n // block) + 4, "flops": 4 * M * E}
    wbytes = 1 if case["kind"] == "fp8" else 2
    active = _active_experts(M, E, topk, s["zipf"])
    nbytes = active * 3 * H * F * wbytes + 2 * M * H * 2  # weights of the experts hit, tokens in, rows out
    flops = 6 * M * topk * H * F
    if case["kind"] == "gate":
        nbytes += 2 * H * E
        flops += 2 * M * H * E
    else:
        nbytes += 4 * M * E
    if case["kind"] == "fp8":
        nbytes += 4 * active * (2 * F + H)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times the distance of the path from the same computation in fp64 on the same operands
    if case["kind"] == "route":  # fp32 softmax weights; ids and routing arrays are whole numbers
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "fp8":  # 2.1e-3 / 1.5e-2, and a code of the activated rows that rounds the other way
        return {"rel": 1.2e-2, "max": 1e-1}
    if case["kind"] == "gate":  # fp16: 3.7e-4 / 1.7e-3
        return {"rel": 1.5e-3, "max": 8e-3}
    return {"rel": 1e-2, "max": 6e-2}  # bf16: 2.3e-3 .. 2.9e-3 / 1.4e-2
