"""The work whose speed this framework is judged by: calls of its public entry points as a program that serves a
quantised language model makes them, over the range of sizes it meets.

  linear   ops.qgemv / ops.qlinear: one projection, y = x @ dequant(W).T, from one decoded token (M = 1) over a batch of
           decoding sequences (M up to a few hundred) to a long prompt (M in the thousands); int4 group-32 and int8
           per-row weights; fp32 results or bf16 ones
  moe      ops.moe_ffn: a mixture-of-experts feed-forward layer, from a few decoding tokens to a prompt, experts in the
           row-major containers or in tile order
  decode   QuantDecoder: one greedy token through the whole model, replayed from its captured graph
  prompt   QuantDecoder.feed: a prompt read into the caches of the same model

Weights, activations and caches are made on the GPU from the seed.
"""
import math

import torch

from chadslab_amd import QWeightInt4G32, QWeightInt8, ops
from chadslab_amd.decoder import DecoderConfig, QuantDecoder, random_weights

DEV = "cuda:0"


def _linear(m, n, k, weight="int4", out="native", **more):
    return dict(more, op="linear", m=m, n=n, k=k, weight=weight, out=out)


def _moe(tokens, h, f, experts, top_k, layout, **more):
    return dict(more, op="moe", tokens=tokens, h=h, f=f, experts=experts, top_k=top_k, layout=layout)


def _model(op, layers=18, d=2048, hq=8, dh=256, ffn=16384, vocab=256000, max_ctx=4096, pos=0, tokens=1, **more):
    return dict(more, op=op, layers=layers, d=d, hq=hq, dh=dh, ffn=ffn, vocab=vocab, max_ctx=max_ctx, pos=pos, tokens=tokens)


def listed():
    return [
        # the smallest projection of the 2B decoder (attention output), one token: launches and host time decide
        _linear(1, 2048, 2048, name="int4 1x2048x2048"),
        # the feed-forward projection of a 7B-sized model, one decoded token (the benchmark's first workload)
        _linear(1, 14336, 4096, name="int4 1x14336x4096"),
        # six sequences decoded together, results wanted in the activations' own type, a width that fits no tile
        _linear(6, 11008, 4096, out="bf16", name="int4 6x11008x4096 bf16"),
        # int8 weights, one decoded token (the benchmark's int8 workload)
        _linear(1, 16384, 2048, weight="int8", name="int8 1x16384x2048"),
        # a serving batch of 48 sequences, one token each: between the decode and the prompt kernels
        _linear(48, 14336, 4096, name="int4 48x14336x4096"),
        # a prompt of 512 tokens (the benchmark's prompt workload)
        _linear(512, 4096, 4096, name="int4 512x4096x4096"),
        # a prompt of a thousand tokens on int8 weights, down projection; no multiple of a tile
        _linear(1000, 4096, 14336, weight="int8", name="int8 1000x4096x14336"),
        # several prompts packed together: the largest product
        _linear(4096, 14336, 4096, name="int4 4096x14336x4096"),
        # four decoding tokens through a mixture of experts kept as it was loaded (row-major)
        _moe(4, 4096, 14336, 8, 2, "rows", name="moe rows 4 tokens"),
        # 256 tokens through the same layer with its experts in tile order (the benchmark's mixture-of-experts workload)
        _moe(256, 4096, 14336, 8, 2, "tiles", name="moe tiles 256 tokens"),
        # one decoded token of the 2B-shaped model at a context of 2048 (the benchmark's decode workload)
        _model("decode", pos=2048, name="decode at 2048"),
        # a prompt of 256 tokens read by the same model
        _model("prompt", tokens=256, name="prompt of 256"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, step, odd=1):
    """lo .. hi, spread over the logarithm: multiples of `step`, one in four of them only of `odd`."""
    step = odd if rng.random() < 0.25 else step
    return max(lo, int(_log(rng, lo, hi) / step + 0.5) * step)


def draw(rng):
    kind = rng.choices(("linear", "moe", "decode", "prompt"), (8, 3, 1, 1))[0]
    if kind == "linear":
        weight = rng.choices(("int4", "int8"), (3, 1))[0]
        m = rng.choices((1, rng.randint(2, 16), int(_log(rng, 17, 256)), int(_log(rng, 256, 4096))), (2, 3, 3, 4))[0]
        n, k = _size(rng, 512, 16384, 128), _size(rng, 512, 16384, 256, 32)
        while m * n * k > 4096 * 14336 * 4096:
            n, k = _size(rng, 512, 16384, 128), _size(rng, 512, 16384, 256, 32)
        return _linear(m, n, k, weight, rng.choice(("native", "bf16")) if m <= 16 else "native")
    if kind == "moe":
        experts = rng.choice((4, 8, 8, 16))
        top_k = rng.choice((1, 2, 2, 4))
        h, f = _size(rng, 1024, 4096, 256, 256), _size(rng, 1024, 14336, 256, 256)
        return _moe(int(_log(rng, 1, 512)), h, f, experts, top_k, rng.choice(("rows", "tiles")))
    hq, dh = rng.choice(((8, 256), (8, 128), (4, 256), (8, 64), (4, 128)))
    d = 256 * rng.randint(2, 8)
    size = dict(layers=rng.randint(2, 12), d=d, hq=hq, dh=dh, ffn=256 * int(d * rng.uniform(3, 8) / 256), vocab=int(_log(rng, 1000, 128000)))
    if kind == "decode":
        return _model("decode", pos=int(_log(rng, 16, 4000)), **size)
    return _model("prompt", tokens=int(_log(rng, 4, 256)), pos=rng.choice((0, rng.randint(1, 1024))), **size)


def _int4(n, k, g):
    """Uniform nibbles with log-normal group scales."""
    packed = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
    scale = torch.exp(torch.randn(n, k // 32, device=DEV, generator=g) * 0.5 - 5.0).to(torch.float16)
    return QWeightInt4G32(packed, scale)


def _int8(n, k, g):
    w = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=DEV, generator=g)
    return QWeightInt8(w, torch.exp(torch.randn(n, device=DEV, generator=g) * 0.5 - 8.0))


def prepare(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    state = {"case": case}
    if case["op"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        state["w"] = (_int8 if case["weight"] == "int8" else _int4)(n, k, g)
        x = torch.randn(m, k, device=DEV, generator=g)
        # decode products on int8 weights take fp32 activations, everything else bf16
        state["x"] = x if case["weight"] == "int8" and m <= ops.GEMV_MAX_M else x.to(torch.bfloat16)
    elif case["op"] == "moe":
        h, f = case["h"], case["f"]
        experts = [(_int4(f, h, g), _int4(f, h, g), _int4(h, f, g)) for _ in range(case["experts"])]
        if case["layout"] == "tiles":
            experts = [tuple(ops.to_tiles(w) for w in triple) for triple in experts]
        state["experts"] = experts
        state["x"] = torch.randn(case["tokens"], h, device=DEV, generator=g).to(torch.bfloat16)
        state["logits"] = torch.randn(case["tokens"], case["experts"], device=DEV, generator=g)
    else:
        cfg = DecoderConfig(n_layers=case["layers"], d=case["d"], hq=case["hq"], dh=case["dh"], ffn=case["ffn"],
                            vocab=case["vocab"], max_ctx=case["max_ctx"])
        dec = QuantDecoder(cfg, random_weights(cfg, seed, DEV), DEV, release_gate_up=True)
        for cache in dec.kcache + dec.vcache:  # the rows an earlier part of the conversation has left
            rows = cache[:case["pos"] * cfg.dh]
            rows.copy_(torch.randn(rows.shape, device=DEV, generator=g))
        dec.capture()
        state["decoder"] = dec
        state["tokens"] = torch.randint(0, cfg.vocab, (case["tokens"],), device=DEV, generator=g).tolist()
    return state


def run(state):
    case = state["case"]
    if case["op"] == "linear":
        if case["out"] == "bf16":
            return ops.qlinear(state["x"], state["w"], out_dtype=torch.bfloat16)
        return ops.qlinear(state["x"], state["w"])
    if case["op"] == "moe":
        return ops.moe_ffn(state["x"], state["logits"], state["experts"], top_k=case["top_k"])
    dec = state["decoder"]
    # The proposed token is the largest of the logits; it is left out of what is compared because two nearly equal
    # logits may change places under another order of summation.
    if case["op"] == "decode":
        dec.set_state(state["tokens"][0], case["pos"])
        dec.graph.replay()
    else:
        dec.feed(state["tokens"], case["pos"])
    return {"logits": dec.logits, "k": dec.kcache, "v": dec.vcache}


def _int4_bytes(n, k):
    return n * (k // 2) + n * (k // 32) * 2


def work(case):
    if case["op"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        weight = n * k + 4 * n if case["weight"] == "int8" else _int4_bytes(n, k)
        x_size = 4 if case["weight"] == "int8" and m <= ops.GEMV_MAX_M else 2
        y_size = 4 if m <= ops.GEMV_MAX_M and case["out"] == "native" else 2
        return {"bytes": weight + m * k * x_size + m * n * y_size, "flops": 2 * m * n * k}
    if case["op"] == "moe":
        t, h, f, e, top_k = case["tokens"], case["h"], case["f"], case["experts"], case["top_k"]
        hit = e * (1 - (1 - top_k / e) ** t)  # experts that some token is sent to, on average
        return {"bytes": hit * 3 * _int4_bytes(f, h) + t * h * 4 + t * e * 4, "flops": 6 * t * top_k * h * f}
    layers, d, hq, dh, ffn = case["layers"], case["d"], case["hq"], case["dh"], case["ffn"]
    pairs = (((hq + 2) * dh, d), (d, hq * dh), (2 * ffn, d), (d, ffn))
    t, pos = case["tokens"], case["pos"]
    rows = t * pos + t * (t + 1) // 2  # (query, key) pairs of one head
    return {"bytes": layers * (sum(_int4_bytes(n, k) for n, k in pairs) + 4 * (pos + t) * dh) + _int4_bytes(case["vocab"], d) + 4 * case["vocab"],
            "flops": layers * (2 * t * sum(n * k for n, k in pairs) + 4 * rows * hq * dh) + 2 * case["vocab"] * d}


def tolerance(case):
    # about four times the distance from the same path evaluated in 64 bits (its roundings to 16 bits kept)
    if case["op"] == "linear":
        if case["m"] <= ops.GEMV_MAX_M:
            if case["out"] == "native":
                return {"rel": 4e-6}  # fp32 sums: 2.6e-7 (int4), 5.7e-7 (int8) at the listed sizes
            return {"rel": 7e-3}  # the same rounded to bf16: 1.65e-3
        if case["weight"] == "int8":
            return {"rel": 7e-3}  # exact weights, bf16 results: 1.66e-3
        return {"rel": 1e-2}  # weights and results rounded to bf16: 2.36e-3
    if case["op"] == "moe":
        return {"rel": 1e-2}  # hidden activations and results in bf16: 3.4e-3 (row-major), 2.1e-3 (tile order)
    # bf16 activations rounded at every layer of a network with random weights, which amplifies every rounding:
    # 1.5e-2 (logits) and 1.4e-2 (deepest caches) over 18 layers, 6e-3 over 4; twice the former is what can be asked
    return {"rel": 3e-2}
