"""The calls that a user of this framework makes, as cases to be timed and compared.

A serving program with speculative decoding calls a MoE layer in three regimes: single-token
decode, verify steps of a few to 128 draft tokens, and prefills of some hundred to 8192
tokens. The shapes are the ones `bench.py` and the tests use: Mixtral-8x7B (bf16, fp16), the
Qwen1.5-MoE and DeepSeek-V2-Lite blocks with a shared expert, the DeepSeek-V2 block with
group-limited routing, and the fp32 layer of hidden 1024. Expert weights are N(0, 0.02), hidden
states N(0, 1); expert pages sit in the pool in a permuted order, as an offload engine leaves
them. Every state has a pool of its own, so that a pass on another state reads cold weights.

`call` names the entry point:
  moe      fused_moe_forward: top-k softmax routing, experts, combine
  stack    stack_fused_moe: experts and combine on the caller's routing
  shared   fused_moe_shared_forward: a block with a shared expert
  grouped  grouped_topk, then stack_fused_moe_shared: group-limited routing
  layer    moe_layer_forward: residual add, RMSNorm, router gate, top-k and the block
"""
import math

import torch

from ae_amd.layers import (fused_moe_forward, fused_moe_shared_forward, grouped_topk,
                           moe_layer_forward, stack_fused_moe, stack_fused_moe_shared)

# hidden, ffn, experts, top-k, shared ffn, gated shared expert, renormalised weights, routed
# scaling factor, expert groups, selectable groups, largest batch drawn
SHAPES = {
    "mixtral": dict(H=4096, I=14336, E=8, k=2, Is=0, gated=False, renorm=True, scale=1.0, ng=1, tg=1, most=8192),
    "qwen15": dict(H=2048, I=1408, E=60, k=4, Is=5632, gated=True, renorm=False, scale=1.0, ng=1, tg=1, most=4096),
    "dsv2lite": dict(H=2048, I=1408, E=64, k=6, Is=2816, gated=False, renorm=False, scale=1.0, ng=1, tg=1, most=4096),
    "dsv2": dict(H=5120, I=1536, E=160, k=6, Is=3072, gated=False, renorm=False, scale=16.0, ng=8, tg=3, most=1024),
    "c1": dict(H=1024, I=2816, E=8, k=2, Is=0, gated=False, renorm=True, scale=1.0, ng=1, tg=1, most=2048),
}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EPS = 1e-5


def listed():
    def case(name, call, shape, tokens, dtype="bf16"):
        return {"name": name, "call": call, "shape": shape, "tokens": tokens, "dtype": dtype}

    return [
        # single-token decode of Mixtral: two experts' weights, 0.7 GB
        case("mixtral_t1", "moe", "mixtral", 1),
        # the headline verify step: 8 sequences x 4 draft tokens
        case("mixtral_t32", "moe", "mixtral", 32),
        # fp16 with routing from the caller (a custom routing function), odd batch
        case("mixtral_stack_f16_t37", "stack", "mixtral", 37, "f16"),
        # the smallest prefill that the solver's performance model is fitted on
        case("mixtral_t400", "moe", "mixtral", 400),
        # the largest prefill of that range
        case("mixtral_t8192", "moe", "mixtral", 8192),
        # a verify step of a many-expert block with a gated shared expert
        case("qwen15_t64", "shared", "qwen15", 64),
        # a prefill of odd length on the same block
        case("qwen15_t1021", "shared", "qwen15", 1021),
        # the smallest call: single-token decode of a small block, where latency counts
        case("dsv2lite_t1", "shared", "dsv2lite", 1),
        # a verify step of the whole post-attention half of a decoder layer
        case("dsv2lite_layer_t32", "layer", "dsv2lite", 32),
        # a prefill of it, of odd length
        case("dsv2lite_layer_t2047", "layer", "dsv2lite", 2047),
        # group-limited routing over 160 experts, verify step
        case("dsv2_grouped_t48", "grouped", "dsv2", 48),
        # the fp32 layer that the CPU baseline runs
        case("c1_f32_t32", "moe", "c1", 32, "f32"),
    ]


def draw(rng):
    shape = rng.choice(["mixtral", "mixtral", "qwen15", "qwen15", "dsv2lite", "dsv2lite", "dsv2", "c1"])
    tokens = int(round(math.exp(rng.uniform(0.0, math.log(SHAPES[shape]["most"])))))
    dtype = "f32" if shape == "c1" else rng.choice(["bf16", "bf16", "f16"])
    calls = {"mixtral": ["moe", "moe", "stack", "layer"], "c1": ["moe", "stack", "layer"], "dsv2": ["grouped"]}
    return {"call": rng.choice(calls.get(shape, ["shared", "shared", "layer"])), "shape": shape,
            "tokens": tokens, "dtype": dtype}


def _normal(g, shape, std, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=g)


def prepare(case, seed):
    s = SHAPES[case["shape"]]
    dtype = DTYPES[case["dtype"]]
    T, H, I, E = case["tokens"], s["H"], s["I"], s["E"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    st = dict(case=case, s=s)
    st["pool"] = _normal(g, (E, 3 * I * H), 0.02, dtype)
    st["slots"] = torch.randperm(E, generator=g, device="cuda")
    st["shared_w"] = _normal(g, (3 * s["Is"] * H,), 0.02, dtype) if s["Is"] else None
    st["x"] = _normal(g, (T, H), 1.0, dtype)
    if case["call"] == "layer":
        # the attention output and the residual stream it is added to
        st["residual"] = _normal(g, (T, H), 1.0, dtype)
        st["norm_w"] = (1.0 + _normal(g, (H,), 0.1, torch.float32)).to(dtype)
        st["gate_w"] = _normal(g, (E, H), 2.0 / math.sqrt(H), dtype)
        st["sgate_w"] = _normal(g, (H,), 1.0 / math.sqrt(H), dtype) if s["gated"] else None
        return st
    if E == 8:
        # a skewed expert load (Zipf, s = 1.2) over the spread a gate of N(0, 0.02) gives
        p = torch.arange(1, E + 1, dtype=torch.float64, device="cuda") ** -1.2
        wg = _normal(g, (E, H), 0.02, dtype)
        st["logits"] = torch.nn.functional.linear(st["x"], wg) + torch.log(p / p.sum()).to(dtype)
    else:
        st["logits"] = _normal(g, (T, E), 2.0, dtype)
    st["sgate"] = _normal(g, (T,), 1.0, dtype) if s["gated"] else None
    if case["call"] == "stack":
        w, ids = torch.softmax(st["logits"].float(), -1).topk(s["k"], dim=-1)
        st["w"], st["ids"] = w / w.sum(-1, keepdim=True), ids.to(torch.int32)
    return st


def run(st):
    s, call = st["s"], st["case"]["call"]
    if call == "moe":
        return fused_moe_forward(st["x"], st["logits"], st["pool"], st["slots"], s["k"], s["renorm"],
                                 inplace=False)
    if call == "stack":
        return stack_fused_moe(st["x"], st["pool"], st["slots"], st["logits"], st["w"], st["ids"],
                               s["renorm"], inplace=False)
    if call == "shared":
        return fused_moe_shared_forward(st["x"], st["logits"], st["pool"], st["slots"], s["k"],
                                        s["renorm"], st["shared_w"], st["sgate"], s["scale"],
                                        inplace=False)
    if call == "grouped":
        w, ids = grouped_topk(st["logits"], s["k"], s["renorm"], s["ng"], s["tg"])
        y = stack_fused_moe_shared(st["x"], st["pool"], st["slots"], w, ids, st["shared_w"],
                                   st["sgate"], s["scale"], inplace=False)
        return y, w, ids
    # the call works in place: the attention hands it new buffers every time
    hidden, residual = st["x"].clone(), st["residual"].clone()
    moe_layer_forward(hidden, residual, st["norm_w"], EPS, st["gate_w"], st["pool"], st["slots"],
                      s["k"], s["renorm"], st["shared_w"], st["sgate_w"], s["scale"])
    return hidden, residual


def work(case):
    s = SHAPES[case["shape"]]
    T, H, I, E, k, Is = case["tokens"], s["H"], s["I"], s["E"], s["k"], s["Is"]
    eb = 4 if case["dtype"] == "f32" else 2
    # experts that some token picks, were the picks uniform
    active = min(E, T * k, E * (1.0 - (1.0 - k / E) ** T))
    weights = 3 * H * (active * I + Is)
    rows = 2 * T * H + T * E
    if case["call"] == "layer":
        weights += (E + 1) * H
        rows += 2 * T * H
    return {"bytes": eb * (weights + rows), "flops": 6.0 * T * H * (k * I + Is)}


def tolerance(case):
    # about four times the difference that another order of the sums makes (the weight-streaming
    # against the tiled kernels on the same inputs): roundings to the activation type that fall
    # the other way. "max": one output's difference over the outputs' root mean square.
    # Measured: bf16 rel 2.3e-4 to 5.5e-4, max 1.9e-2; fp16 1.1e-4, 1.9e-3; fp32 1.1e-6, 5.5e-6.
    return {"bf16": {"rel": 2e-3, "max": 0.07}, "f16": {"rel": 5e-4, "max": 8e-3},
            "f32": {"rel": 5e-6, "max": 2.5e-5}}[case["dtype"]]


def _picks(scores, k):
    """The k best per row, ties to the lower index."""
    return torch.sort(scores, dim=-1, descending=True, stable=True).indices[:, :k]


def exact(case, seed):
    st = prepare(case, seed)
    s, call = st["s"], case["call"]
    H, I, k = s["H"], s["I"], s["k"]
    x = st["x"].double()
    residual = sgate = None
    if call == "layer":
        residual = x + st["residual"].double()
        xn = residual * torch.rsqrt(residual.square().mean(-1, keepdim=True) + EPS) * st["norm_w"].double()
        # the routing is decided on the normalised states and logits as they are stored
        x = xn.to(st["x"].dtype).double()
        logits = (x @ st["gate_w"].double().t()).to(st["x"].dtype).double()
        x = xn
        if s["gated"]:
            sgate = xn @ st["sgate_w"].double()
    else:
        logits = st["logits"].double()
        if s["gated"]:
            sgate = st["sgate"].double()
    if call == "stack":
        w, ids = st["w"].double(), st["ids"].long()
    else:
        p = torch.softmax(logits, -1)
        choice = p
        if call == "grouped":
            best = p.view(p.shape[0], s["ng"], -1).amax(-1)
            open_ = torch.zeros_like(best, dtype=torch.bool).scatter_(1, _picks(best, s["tg"]), True)
            choice = p.masked_fill(~open_.repeat_interleave(p.shape[1] // s["ng"], 1), -1.0)
        ids = _picks(choice, k)
        w = p.gather(1, ids)
        if s["renorm"]:
            w = w / w.sum(-1, keepdim=True)

    def mlp(page, rows, ffn):
        gate, up, down = (page[i * ffn * H:(i + 1) * ffn * H] for i in range(3))
        a = torch.nn.functional.silu(rows @ gate.double().view(ffn, H).t()) * (rows @ up.double().view(ffn, H).t())
        return a @ down.double().view(H, ffn).t()

    y = torch.zeros_like(x)
    for e in range(s["E"]):
        t, j = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            y.index_add_(0, t, mlp(st["pool"][st["slots"][e]], x[t], I) * w[t, j].unsqueeze(1))
    y = y * s["scale"]
    if s["Is"]:
        sh = mlp(st["shared_w"], x, s["Is"])
        y = y + (torch.sigmoid(sgate).unsqueeze(1) * sh if s["gated"] else sh)
    if call == "grouped":
        return y, w, None
    return (y, residual) if call == "layer" else y
