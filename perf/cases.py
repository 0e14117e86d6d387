"""The calls this library's users make, as timed cases: decode steps, prompt batches and dense MLPs over the layer
shapes of this repository (bench.py, mference_amd/fused_shapes.json) and over shapes nobody tuned for.

  listed()         the cases with names
  draw(rng)        one more case of the same ranges
  prepare(case, seed)  weights, inputs, handles and buffers a program holds before the call
  run(state)       one pass through the public operators
  work(case)       bytes and operations a pass cannot do without
  tolerance(case)  how far two correct implementations may differ
"""
import functools

import numpy as np
import torch

from mference_amd import operators as ops

# Layer shapes.  bits 1: ternary.  route: who routes -- the layer's own router, or a family router called in front of
# it whose result the layer reads.  fs: width of the 4-bit shared expert.  mlp8: width of the 8-bit dense MLP that runs beside the experts.
MODELS = {
    # the 4-bit layer of the benchmark: 256 small experts and a gated shared expert
    "qwen": dict(d=2048, f=512, e=256, k=8, fs=512, bits=4, route="own", mlp8=0),
    # the large 2-bit layer: sqrt-softplus routing, 4-bit shared expert
    "large2bit": dict(d=4096, f=2048, e=256, k=6, fs=2048, bits=2, route="sqrtsoftplus", mlp8=0),
    # the two ternary layers: full-softmax router, no shared expert
    "ternary": dict(d=2048, f=1024, e=64, k=8, fs=0, bits=1, route="own", mlp8=0),
    "maple": dict(d=2048, f=512, e=256, k=8, fs=0, bits=1, route="own", mlp8=0),
    # 8-bit router rows in front, 4-bit experts of a width that is no multiple of 128, an 8-bit dense MLP beside them
    "gemma": dict(d=2816, f=704, e=128, k=8, fs=0, bits=4, route="gemma", mlp8=2112),
}
# the dense SwiGLU MLP of the benchmark
DENSE = dict(d=5120, f=17408)


def _moe_case(kind, model, t, **more):
    return dict(kind=kind, model=model, t=t, **MODELS.get(model, {}), **more)


def listed():
    return [
        # one token through a stack of small layers of a shape no kernel was written for: launches and host work
        dict(_moe_case("decode", "other", 1, d=1024, f=384, e=48, k=4, fs=384, bits=4, route="own", mlp8=0, layers=4,
                       form="plain", replay=False), name="token-small"),
        # one token through the benchmark's layers with residual add and norm in front, called layer by layer
        dict(_moe_case("decode", "qwen", 1, layers=8, form="normed", replay=False), name="token-qwen"),
        # five sequences decoded together, the stack replayed from a captured graph as a serving loop does
        dict(_moe_case("decode", "qwen", 5, layers=8, form="plain", replay=True), name="batch-qwen-replay"),
        # one token through the large 2-bit layers, routed by their family's router
        dict(_moe_case("decode", "large2bit", 1, layers=3, form="plain", replay=False), name="token-2bit"),
        # one token through the ternary layers
        dict(_moe_case("decode", "maple", 1, layers=12, form="plain", replay=False), name="token-ternary"),
        # one token through layers with an 8-bit router in front and an 8-bit MLP beside the experts
        dict(_moe_case("decode", "gemma", 1, layers=8, form="plain", replay=False), name="token-gemma"),
        # a long prompt chunk through one layer, from the tiled pool
        dict(_moe_case("prompt", "qwen", 2048, tiled=True, narrow=False), name="prompt-qwen-2048"),
        # a short prompt of a ragged length, from the pool as loaded
        dict(_moe_case("prompt", "qwen", 93, tiled=False, narrow=False), name="prompt-qwen-93"),
        # a medium prompt through the large 2-bit layer
        dict(_moe_case("prompt", "large2bit", 777, tiled=True, narrow=False), name="prompt-2bit-777"),
        # a medium prompt through the layer whose expert width is no multiple of 128
        dict(_moe_case("prompt", "gemma", 300, tiled=False, narrow=False), name="prompt-gemma-300"),
        # four rows through the dense MLP: a draft of three tokens being verified
        dict(kind="mlp", t=4, bits=4, sets=2, **DENSE, name="mlp-verify"),
        # a prompt block through the dense MLP
        dict(kind="mlp", t=150, bits=4, sets=2, **DENSE, name="mlp-block-150"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _other(rng):
    """a layer shape nobody wrote a kernel for: widths are multiples of the quantization group"""
    bits = rng.choice([4, 4, 2, 1])
    e = 32 * rng.randint(1, 8) if bits == 1 else rng.randint(12, 200)
    f = 64 * _log_int(rng, 3, 24)
    return dict(d=64 * _log_int(rng, 8, 56), f=f, e=e, k=rng.randint(2, 8), fs=0 if bits == 1 else rng.choice([0, f]), bits=bits, route="own", mlp8=0)


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "mlp"])
    if kind == "mlp":
        d, f = rng.choice([(DENSE["d"], DENSE["f"]), (64 * _log_int(rng, 16, 80), 64 * _log_int(rng, 32, 200))])
        return dict(kind="mlp", t=rng.choice([1, rng.randint(2, 8), _log_int(rng, 9, 512)]), bits=rng.choice([4, 4, 4, 2]), sets=2, d=d, f=f)
    model = rng.choice(["qwen", "qwen", "large2bit", "ternary", "maple", "gemma", "other", "other"])
    shape = _other(rng) if model == "other" else {}
    if kind == "decode":
        c = _moe_case("decode", model, rng.choice([1, rng.randint(1, 8)]), **shape)
        own = c["route"] == "own"
        return dict(c, layers=rng.randint(2, 3) if model == "large2bit" else rng.randint(4, 12), form=rng.choice(["plain", "normed"]) if own else "plain",
                    replay=rng.random() < 0.3)
    c = _moe_case("prompt", model, 1, **shape)
    most = work(_of(listed(), "prompt-2bit-777"))["flops"]
    top = 4096
    while work(dict(c, t=top))["flops"] > most:
        top = int(top * 0.9)
    matrix = c["d"] % 128 == 0 and c["f"] % 128 == 0
    return dict(c, t=_log_int(rng, 9, top), tiled=matrix and rng.random() < 0.5, narrow=matrix and rng.random() < 0.25)


def _of(cases, name):
    return next(c for c in cases if c["name"] == name)


# ------------------------------------------------------------------ preparation

_CTX = []


def _context():
    if not _CTX:
        _CTX.append(ops.MetalContext(0))
    return _CTX[0]


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


def _bf16(t):
    return t.to(torch.bfloat16)


def _quantized(gen, rows, cols, bits):
    """N(0, 0.02) weights, quantized; ternary: codes {0,1,2} with p = .25/.5/.25 and a scale per 64"""
    if bits != 1:
        return ops.Quantization(_context()).quantize_affine(_randn(gen, rows, cols) * 0.02, bits)
    u = torch.rand((rows, cols // 4, 4), generator=gen, device="cuda")
    c = (u >= 0.25).to(torch.uint8) + (u >= 0.75).to(torch.uint8)
    packed = (c[..., 0] | (c[..., 1] << 2) | (c[..., 2] << 4) | (c[..., 3] << 6)).contiguous()
    scales = _bf16(_randn(gen, rows, cols // 64).abs() * 0.02 + 1e-3)
    return ops.QuantizedTensor(packed, scales, -scales, 1, rows, cols)


def _layer(case, gen, skewed):
    """one resident layer: (weights the layer call takes, what the family router and the 8-bit MLP take)"""
    d, f, e, bits = case["d"], case["f"], case["e"], case["bits"]
    off, _, stride = ops.expert_blob_layout(d, f, bits)
    pool = torch.zeros((e, stride), dtype=torch.uint8, device="cuda")
    for name, rows, cols in (("gate", f, d), ("up", f, d), ("down", d, f)):
        q = _quantized(gen, e * rows, cols, bits)
        parts = [("w", q.packed), ("s", q.scales)] + ([("b", q.biases)] if bits != 1 else [])
        for s, v in parts:
            v = v.view(torch.uint8).view(e, -1)
            at = getattr(off, "%s_%s" % (name, s))
            pool[:, at:at + v.shape[1]] = v
        del q
    router = _randn(gen, e, d) * 0.02
    if skewed:  # uneven loads: a bias per expert, carried by a last feature of x that is one
        router[:, -1] = _randn(gen, e) * 1.5
    more = {}
    if case["route"] == "gemma":
        q = ops.Quantization(_context()).quantize_affine(router, 8)
        more["router8"] = q
        more["effective"] = _bf16(1.0 + 0.1 * _randn(gen, d))
        more["per_expert"] = _bf16(1.0 + 0.1 * _randn(gen, e))
    elif case["route"] == "sqrtsoftplus":
        more["router_w"] = _bf16(router)
        more["correction"] = 0.1 * _randn(gen, e)
    if case["mlp8"]:
        m = case["mlp8"]
        more["mlp8"] = [ops.Quantization(_context()).quantize_affine(_randn(gen, r, c) * 0.02, 8) for r, c in ((m, d), (m, d), (d, m))]
    shared = sg = None
    if case["fs"]:
        fs = case["fs"]
        shared = [_quantized(gen, r, c, 4) for r, c in ((fs, d), (fs, d), (d, fs))]
        sg = _bf16(_randn(gen, d) * 0.02)
    lw = ops.MoELayerWeights(_bf16(router) if case["route"] == "own" else None, pool, off, shared, sg)
    return lw, more


def _handle(case):
    ternary = case["bits"] == 1
    return ops.MoE(_context(), case["d"], case["f"], case["e"], case["k"], bits=case["bits"], shared_f=case["fs"], shared_bits=4,
                   maple_rounding=ternary, router_mode=ops.ROUTER_FULL_SOFTMAX if ternary else ops.ROUTER_TOPK_SOFTMAX)


def _route_buffers(case, n):
    t, k, e, d = case["t"], case["k"], case["e"], case["d"]
    b = {"idx": torch.zeros((n, t, k), dtype=torch.int32, device="cuda"), "w": torch.zeros((n, t, k), dtype=torch.float32, device="cuda")}
    if case["route"] != "own":
        b["logits"] = torch.zeros((t, e), dtype=torch.float32, device="cuda")
        b["fam"] = ops.FamilyRouters(_context())
    if case["mlp8"]:
        b["op8"] = ops.SharedExpertInt8(_context())
        b["act8"] = torch.zeros((t, case["mlp8"]), dtype=torch.bfloat16, device="cuda")
        b["y8"] = torch.zeros((n, t, d), dtype=torch.bfloat16, device="cuda")
    return b


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1_000_003 * int(seed) + 17)
    t, d = case["t"], case["d"]
    s = {"case": case}
    if case["kind"] == "mlp":
        f, n = case["f"], case["sets"]
        s["sets"] = [[_quantized(gen, r, c, case["bits"]) for r, c in ((f, d), (f, d), (d, f))] for _ in range(n)]
        s["op"] = ops.SharedExpertInt4(_context())
        s["x"] = _bf16(_randn(gen, n, t, d))
        s["y"] = torch.zeros((n, t, d), dtype=torch.bfloat16, device="cuda")
        s["scratch"] = torch.zeros(max(s["op"].scratch_bytes(d, f, t), t * f * 2), dtype=torch.uint8, device="cuda").view(torch.bfloat16)
        return s
    s["moe"] = _handle(case)
    if case["kind"] == "prompt":
        lw, more = _layer(case, gen, True)
        s.update(more, lw=lw, x=_bf16(_randn(gen, t, d)), y=torch.zeros((t, d), dtype=torch.bfloat16, device="cuda"), **_route_buffers(case, 1))
        s["x"][:, -1] = 1.0
        if case["tiled"]:
            lw.experts_tiled = s["moe"].tile_experts(lw.experts, lw.offsets)
        if case["narrow"]:
            s["moe"].set_prefill_route_rounding(True)
        s["ws"] = torch.empty(max(s["moe"].prefill_workspace_bytes(t), 16), dtype=torch.uint8, device="cuda")
        return s
    n = case["layers"]
    s["layers"] = [_layer(case, gen, False) for _ in range(n)]
    s.update(_route_buffers(case, n), x=_bf16(_randn(gen, n, t, d)), y=torch.zeros((n, t, d), dtype=torch.bfloat16, device="cuda"))
    if case["form"] == "normed":
        s["norm"] = _bf16(1.0 + 0.1 * _randn(gen, n, d))
        s["delta"] = _bf16(_randn(gen, n, t, d) * 0.5)
        s["hidden"] = torch.empty_like(s["x"])
    if case["replay"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = _step(s)
    return s


# ------------------------------------------------------------------ one pass

def _route(s, more, x, i):
    c = s["case"]
    if c["route"] == "gemma":
        q = more["router8"]
        s["fam"].encode_router_gemma4(q.packed, q.scales, q.biases, x, more["effective"], more["per_expert"], s["idx"][i], s["w"][i],
                                      c["e"], c["d"], c["k"], s["logits"], t=c["t"])
    elif c["route"] == "sqrtsoftplus":
        s["fam"].encode_router_top_k(more["router_w"], x, more["correction"], s["idx"][i], s["w"][i], c["e"], c["d"], 1.5, s["logits"],
                                     top_k=c["k"], t=c["t"])


def _beside(s, more, x, i):
    if s["case"]["mlp8"]:
        g, u, dn = more["mlp8"]
        s["op8"].encode(x, g, u, dn, s["y8"][i], s["act8"], t=s["case"]["t"])


def _outputs(s):
    return {k: s[k] for k in ("y", "idx", "w", "hidden", "y8") if k in s}


def _step(s):
    """one decode step: every layer on rows of its own, as attention leaves them between the layers"""
    c, moe, t = s["case"], s["moe"], s["case"]["t"]
    if c["form"] == "normed":
        s["hidden"].copy_(s["x"])
    for i, (lw, more) in enumerate(s["layers"]):
        if c["form"] == "normed":
            moe.encode_decode_layer_normed(lw, s["hidden"][i], s["norm"][i], s["y"][i], t=t, delta=s["delta"][i], out_indices=s["idx"][i],
                                           out_weights=s["w"][i])
            continue
        x = s["x"][i]
        _route(s, more, x, i)
        moe.encode_decode_layer(lw, x, s["y"][i], t=t, out_indices=s["idx"][i], out_weights=s["w"][i])
        _beside(s, more, x, i)
    return _outputs(s)


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "mlp":
        for i, (g, u, dn) in enumerate(s["sets"]):
            s["op"].encode(s["x"][i], g, u, dn, s["y"][i], s["scratch"], t=c["t"])
        return {"y": s["y"]}
    if c["kind"] == "prompt":
        _route(s, s, s["x"], 0)
        s["moe"].encode_prefill_layer(s["lw"], s["x"], s["y"], c["t"], workspace=s["ws"], out_indices=s["idx"][0], out_weights=s["w"][0])
        _beside(s, s, s["x"], 0)
        return _outputs(s)
    if c["replay"]:
        s["graph"].replay()
        return s["out"]
    return _step(s)


# ------------------------------------------------------------------ what a pass needs

def _tensor_bytes(rows, cols, bits):
    """codes, and a 2-byte scale and bias per group of 64 (ternary: the scale alone)"""
    return rows * cols * (2 if bits == 1 else bits) // 8 + rows * (cols // 64) * (2 if bits == 1 else 4)


@functools.lru_cache(maxsize=None)
def _live(e, k, t, skewed):
    """experts that a batch of t tokens touches, for logits like the ones prepare() makes"""
    r = np.random.RandomState(1)
    bias = r.standard_normal(e) * 1.5 * skewed
    top = np.argpartition(-(r.standard_normal((min(t, 4096), e)) + bias), k - 1, axis=1)[:, :k] if k < e else np.arange(e)
    return len(np.unique(top))


def work(case):
    t, d, f = case["t"], case["d"], case["f"]
    if case["kind"] == "mlp":
        n = case["sets"]
        return {"bytes": n * (2 * _tensor_bytes(f, d, case["bits"]) + _tensor_bytes(d, f, case["bits"]) + 4 * t * d), "flops": n * 6 * t * d * f}
    e, k, fs, m = case["e"], case["k"], case["fs"], case["mlp8"]
    n = case.get("layers", 1)
    one = 2 * _tensor_bytes(f, d, case["bits"]) + _tensor_bytes(d, f, case["bits"])
    b = _live(e, k, t, case["kind"] == "prompt") * one + (_tensor_bytes(e, d, 8) if case["route"] == "gemma" else 2 * e * d)
    b += 4 * t * d + 8 * t * k
    if fs:
        b += 2 * _tensor_bytes(fs, d, 4) + _tensor_bytes(d, fs, 4) + 2 * d
    if m:
        b += 3 * _tensor_bytes(m, d, 8) + 2 * t * d
    if case.get("form") == "normed":
        b += 4 * t * d + 2 * d
    return {"bytes": n * b, "flops": n * (2 * t * e * d + 6 * t * d * (k * f + fs + m))}


def tolerance(case):
    # bf16 results of bf16 activations in between: an activation that lands on the other side of a rounding boundary
    # moves a result by parts of its last place.  The routing is whole numbers and has no slack.
    return {"rel": 4e-3, "max": 3e-2, "differ": 0.0}
