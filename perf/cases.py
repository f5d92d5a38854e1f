"""The work that users of this package have it do, as cases to measure.

A case is a dict of plain values; its ``kind`` names the entry point and the rest are sizes and options:

* ``w4``       packed-int4 linears (``W4A16Linear``), group 128, from one decode token to a prefill;
* ``w8``       int8 linears (``SmoothQuantLinear``, the fake-quant rule of its default);
* ``mlp``      the serving runtime's norm + dense W8A8 MLP (``add_rms_norm_forward`` -> ``dense_mlp_w8a8``);
* ``experts``  packed int8 experts (``SmoothQuantPackedMoeExperts``, the fake-quant rule of its default);
* ``fused``    the serving runtime's expert chain (``fused_experts_w8a8``, fp32 scales);
* ``decode``   one greedy step of a W4A16 decoder stack (``W4Decoder.decode_step``);
* ``prefill``  the prompt pass of the same stack (``W4Decoder.prefill``).

Weights are what a loaded checkpoint holds: codes of bell-shaped weights with the scales that go with them.
Calls of a few rows run as a serving loop runs them, captured once into a HIP graph and replayed
(``graph``); the others are called as they are.  ``layers`` linears or blocks of one shape follow each
other in a pass where one alone would stay in the caches, which it does not inside a model.
"""
import math
from types import SimpleNamespace

import torch

HEAD = 128  # the head size of the decoder stacks
GROUP = 128  # int4 weights per scale
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # the smallest call: one token through one square int4 linear, called eagerly (launch and call latency)
        {"name": "w4-fp16-1", "kind": "w4", "dtype": "fp16", "rows": 1, "inp": 4096, "out": 4096, "bias": False, "layers": 1,
         "graph": False},
        # a decode batch through the gate or up projections of a 70B-shaped model, in bf16 as it is served
        {"name": "w4-bf16-16", "kind": "w4", "dtype": "bf16", "rows": 16, "inp": 8192, "out": 28672, "bias": False, "layers": 2,
         "graph": True},
        # a short prompt (or a chunk of one): odd row count, biases, sizes that are not powers of two
        {"name": "w4-fp16-77", "kind": "w4", "dtype": "fp16", "rows": 77, "inp": 5120, "out": 13824, "bias": True, "layers": 4,
         "graph": False},
        # a few sequences decoded through a smoothed 7B-shaped up projection in bf16, the weights' own dtype
        {"name": "w8-bf16-8", "kind": "w8", "dtype": "bf16", "rows": 8, "inp": 4096, "out": 11008, "bias": False, "layers": 4,
         "graph": True},
        # a long prompt through the same projection in fp16
        {"name": "w8-fp16-4096", "kind": "w8", "dtype": "fp16", "rows": 4096, "inp": 4096, "out": 11008, "bias": False,
         "layers": 1, "graph": False},
        # a ragged prompt chunk in bf16 with a bias
        {"name": "w8-bf16-1000", "kind": "w8", "dtype": "bf16", "rows": 1000, "inp": 5120, "out": 13824, "bias": True,
         "layers": 1, "graph": False},
        # the serving runtime's norm and MLP for a mid-sized batch of decode tokens
        {"name": "mlp-bf16-200", "kind": "mlp", "dtype": "bf16", "rows": 200, "inp": 4096, "inter": 11008, "layers": 3,
         "graph": True},
        # the Mixtral-shaped experts module on 512 tokens, top-2 of 8
        {"name": "experts-fp16-512", "kind": "experts", "dtype": "fp16", "rows": 512, "experts": 8, "top": 2, "inp": 4096,
         "inter": 14336, "layers": 1, "graph": False},
        # the serving runtime's experts of the same shape on a decode batch
        {"name": "fused-bf16-48", "kind": "fused", "dtype": "bf16", "rows": 48, "experts": 8, "top": 2, "inp": 4096,
         "inter": 14336, "layers": 1, "graph": True},
        # one sequence decoded by a 7B-shaped stack (four of its layers and its head), odd context length
        {"name": "decode-1", "kind": "decode", "rows": 1, "context": 2117, "heads": 32, "kv": 32, "inter": 11008,
         "vocab": 32000, "layers": 4, "graph": True},
        # sixteen sequences of 4096 tokens decoded by a 70B-shaped stack (two of its layers and its head)
        {"name": "decode-16", "kind": "decode", "rows": 16, "context": 4096, "heads": 64, "kv": 8, "inter": 28672,
         "vocab": 128256, "layers": 2, "graph": True},
        # the prompt of a 7B-shaped stack: 2048 tokens through two of its layers, then the head
        {"name": "prefill-2048", "kind": "prefill", "rows": 2048, "heads": 32, "kv": 32, "inter": 11008, "vocab": 32000,
         "layers": 2, "graph": False},
    ]


def _log_int(rng, lo, hi, step=1):
    """A whole number spread over the logarithm of ``lo .. hi``, a multiple of ``step``."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["w4", "w4", "w8", "w8", "mlp", "experts", "fused", "decode", "prefill"])
    if kind in ("w4", "w8"):
        rows = _log_int(rng, 1, 4096)
        inp, out = _log_int(rng, 1024, 8192, 128), _log_int(rng, 1024, 28672, 8)
        if rng.random() < 0.15:  # a down projection: long reductions
            inp, out = _log_int(rng, 11008, 28672, 128), _log_int(rng, 1024, 8192, 8)
        rows = max(1, min(rows, int(4e11 / (2 * inp * out))))
        return {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "rows": rows, "inp": inp, "out": out,
                "bias": rng.random() < 0.3, "layers": 1 if rows > 256 else 3, "graph": rows <= 64}
    if kind == "mlp":
        rows = _log_int(rng, 1, 2048)
        return {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "rows": rows, "inp": _log_int(rng, 1024, 8192, 128),
                "inter": _log_int(rng, 1024, 14336, 128), "layers": 1 if rows > 256 else 2, "graph": rows <= 256}
    if kind in ("experts", "fused"):
        rows, experts = _log_int(rng, 1, 1024), rng.choice([4, 8, 16, 32])
        inp = _log_int(rng, 1024, 4096, 128)
        inter = _log_int(rng, 512, min(14336, int(1.4e9 / (3 * experts * inp))), 64)
        return {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "rows": rows, "experts": experts,
                "top": rng.choice([1, 2, 4]), "inp": inp, "inter": inter, "layers": 1, "graph": rows <= 64}
    kv = rng.choice([4, 8, 16, 32])
    heads = kv * rng.choice([g for g in (1, 2, 4, 8) if 16 <= kv * g <= 64])
    inter = _log_int(rng, 4096, min(28672, 384 * heads), 256)
    if kind == "decode":
        rows = _log_int(rng, 1, 48)
        return {"kind": kind, "rows": rows, "context": min(_log_int(rng, 64, 4096), 2 ** 19 // (rows * kv)), "heads": heads, "kv": kv,
                "inter": inter, "vocab": rng.choice([32000, 64000]), "layers": 2, "graph": True}
    return {"kind": kind, "rows": _log_int(rng, 65, 2048), "heads": min(heads, 32), "kv": min(kv, 32), "inter": min(inter, 14336),
            "vocab": 32000, "layers": 1, "graph": False}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _w4_weight(n, k, dtype, gen):
    """``(packed int32 [N, K/8], scales [N, K/128], zeros [N, K/128])`` of an asymmetric int4 weight of std about 0.02."""
    u = (torch.randn(n, k, generator=gen, device="cuda", dtype=torch.float16) * 2.6 + 7.5).round_().clamp_(0, 15)
    u = u.to(torch.int32).view(n, k // 8, 8)
    packed = u[:, :, 0].clone()
    for j in range(1, 8):
        packed |= u[:, :, j] << (4 * j)
    g = k // GROUP
    scales = (0.0077 * (0.8 + 0.4 * torch.rand(n, g, generator=gen, device="cuda"))).to(dtype)
    zeros = (7.5 + torch.randn(n, g, generator=gen, device="cuda") * 0.8).round_().clamp_(0, 15).to(dtype)
    return packed.contiguous(), scales, zeros


def _w8_weight(shape, dtype, gen):
    """``(codes int8, scales fp32 per row, exact in dtype)`` of a weight of std about 0.02."""
    codes = torch.empty(shape, dtype=torch.int8, device="cuda")
    flat = codes.view(-1, shape[-1])
    step = max(1, (1 << 26) // shape[-1])
    for i in range(0, flat.shape[0], step):
        part = flat[i:i + step]
        part.copy_((torch.randn(part.shape, generator=gen, device="cuda", dtype=torch.float16) * 30.0).round_().clamp_(-127, 127))
    scales = (0.02 / 30.0 * (0.8 + 0.4 * torch.rand(shape[:-1], generator=gen, device="cuda"))).to(dtype).float()
    return codes, scales


def _acts(rows, k, dtype, gen):
    """Activations ~ N(0, 1) with 1% of the channels three times as large (smoothed outliers)."""
    x = torch.randn(rows, k, generator=gen, device="cuda")
    x[:, ::100] *= 3.0
    return x.to(dtype)


def _routing(rows, experts, top, gen):
    """Top-k ids int32 and weights fp32 (summing to one) of N(0, 1) router logits."""
    p = torch.softmax(torch.randn(rows, experts, generator=gen, device="cuda"), -1)
    w, ids = torch.topk(p, top, dim=-1)
    return ids.contiguous(), (w / w.sum(-1, keepdim=True)).contiguous()


def _weights(case, seed):
    """The tensors of a case, by name: what a checkpoint and a prompt give."""
    gen, kind = _gen(seed), case["kind"]
    if kind in ("decode", "prefill"):
        h, q, kv, inter = case["heads"] * HEAD, case["heads"], case["kv"], case["inter"]
        dt = torch.float16
        layers = []
        for _ in range(case["layers"]):
            layers.append({"ln1": (1.0 + 0.1 * torch.randn(h, generator=gen, device="cuda")).to(dt),
                           "ln2": (1.0 + 0.1 * torch.randn(h, generator=gen, device="cuda")).to(dt),
                           "qkv": _w4_weight((q + 2 * kv) * HEAD, h, dt, gen), "o": _w4_weight(h, h, dt, gen),
                           "gate_up": _w4_weight(2 * inter, h, dt, gen), "down": _w4_weight(h, inter, dt, gen)})
        t = {"layers": layers, "lm_head": _w4_weight(case["vocab"], h, dt, gen),
             "embed": torch.randn(case["vocab"], h, generator=gen, device="cuda").to(dt)}
        if kind == "decode":
            shape = (case["layers"], case["rows"], kv, case["context"] + 1, HEAD)
            t["k"] = torch.randn(shape, generator=gen, device="cuda", dtype=dt)
            t["v"] = torch.randn(shape, generator=gen, device="cuda", dtype=dt)
            t["tokens"] = torch.randint(0, case["vocab"], (case["rows"],), generator=gen, device="cuda")
        else:
            t["tokens"] = torch.randint(0, case["vocab"], (1, case["rows"]), generator=gen, device="cuda")
        return t
    dt = DTYPES[case["dtype"]]
    t = {"x": _acts(case["rows"], case["inp"], dt, gen), "layers": []}
    if kind in ("experts", "fused"):
        t["ids"], t["topw"] = _routing(case["rows"], case["experts"], case["top"], gen)
    for _ in range(case["layers"]):
        if kind == "w4":
            w = _w4_weight(case["out"], case["inp"], dt, gen)
        elif kind == "w8":
            w = _w8_weight((case["out"], case["inp"]), dt, gen)
        elif kind == "mlp":
            w = (_w8_weight((2 * case["inter"], case["inp"]), dt, gen), _w8_weight((case["inp"], case["inter"]), dt, gen),
                 (1.0 + 0.1 * torch.randn(case["inp"], generator=gen, device="cuda")).to(dt),
                 _acts(case["rows"], case["inp"], dt, gen))
        else:
            e = case["experts"]
            w = (_w8_weight((e, 2 * case["inter"], case["inp"]), dt, gen),
                 _w8_weight((e, case["inp"], case["inter"]), dt, gen))
        b = (0.1 * torch.randn(case["out"], generator=gen, device="cuda")).to(dt) if case.get("bias") else None
        t["layers"].append((w, b))
    return t


# ---------------------------------------------------------------- the calls
def _linears(case, t):
    """One call per linear of the case, as a closure over the modules that hold the weights."""
    from mindpipe_amd.smoothquant import SmoothQuantLinear
    from mindpipe_amd.w4a16 import W4A16Linear
    dt, mods = DTYPES[case["dtype"]], []
    for w, b in t["layers"]:
        if case["kind"] == "w4":
            m = W4A16Linear(case["inp"], case["out"], GROUP, b is not None, True, dtype=dt, device="cuda")
            m.weight_packed, m.weight_scale, m.weight_zero_point = w
        else:
            m = SmoothQuantLinear(case["inp"], case["out"], b is not None, dtype=dt).to("cuda")
            m.weight, m.weight_scale = w
        if b is not None:
            m.bias = b
        mods.append(m)
    return lambda: [m(t["x"]) for m in mods]


def _mlp(case, t):
    from mindpipe_amd import runtime
    method, dt, blocks = runtime.W8A8DynamicLinearMethod(), DTYPES[case["dtype"]], []
    for (w13, w2, ln, res), _ in t["layers"]:
        pair = []
        for q, s in (w13, w2):
            layer = SimpleNamespace(weight=torch.nn.Parameter(q, requires_grad=False), quant_method=method, params_dtype=dt,
                                    weight_scale=torch.nn.Parameter(s.unsqueeze(-1), requires_grad=False))
            method.process_weights_after_loading(layer)
            pair.append(layer)
        runtime.prepare_dense_mlp_w8a8(*pair)
        blocks.append((SimpleNamespace(weight=ln, variance_epsilon=1e-5), res, *pair))

    def call():
        x, out = t["x"], []
        for norm, res, gate_up, down in blocks:
            y, rsum = runtime.add_rms_norm_forward(norm, x, res, gate_up)
            out += [runtime.dense_mlp_w8a8(gate_up, down, y), rsum]
        return out
    return call


def _experts(case, t):
    from mindpipe_amd import runtime
    from mindpipe_amd.smoothquant import SmoothQuantPackedMoeExperts
    (w13, w2), _ = t["layers"][0]
    if case["kind"] == "experts":
        # a module whose buffers the checkpoint then fills
        dt = DTYPES[case["dtype"]]
        m = SmoothQuantPackedMoeExperts(torch.zeros(1, 128, 64, device="cuda", dtype=dt),
                                        torch.zeros(1, 64, 64, device="cuda", dtype=dt), torch.nn.SiLU())
        m.num_experts, m.hidden_dim, m.intermediate_dim = case["experts"], case["inp"], case["inter"]
        (m.gate_up_proj, m.gate_up_scale), (m.down_proj, m.down_scale) = w13, w2
        return lambda: m(t["x"], t["ids"], t["topw"])
    layer = SimpleNamespace(**{f"{n}_{a}": torch.nn.Parameter(v, requires_grad=False) for n, w in (("w13", w13), ("w2", w2))
                               for a, v in (("weight", w[0]), ("weight_scale", w[1].unsqueeze(-1)))})
    method = runtime.W8A8DynamicFusedMoEMethod(DTYPES[case["dtype"]])
    method.process_weights_after_loading(layer)
    ids = t["ids"].to(torch.int32)
    return lambda: runtime.fused_experts_w8a8(t["x"], layer.w13_weight, layer.w13_weight_scale_fp32, layer.w2_weight,
                                              layer.w2_weight_scale_fp32, t["topw"], ids, output_dtype=t["x"].dtype)


def _stack(case, t):
    from mindpipe_amd.decoder import DecoderConfig, W4Decoder
    decode = case["kind"] == "decode"
    cfg = DecoderConfig(layers=case["layers"], hidden=case["heads"] * HEAD, heads=case["heads"], kv_heads=case["kv"],
                        ffn=case["inter"], vocab=case["vocab"], group=GROUP)
    d = W4Decoder(cfg, case["rows"] if decode else 1, case["context"] + 1 if decode else case["rows"])
    d.embed = t["embed"]
    for have, new in zip(d.layers, t["layers"]):
        have["ln1"], have["ln2"] = new["ln1"], new["ln2"]
        for n in ("qkv", "o", "gate_up", "down"):
            have[n].packed, have[n].scales, have[n].zeros = new[n]
    d.lm_head.packed, d.lm_head.scales, d.lm_head.zeros = t["lm_head"]
    if decode:
        d.k_cache, d.v_cache = t["k"], t["v"]
        at = torch.tensor([case["context"]], device="cuda", dtype=torch.int64)
        return lambda: {"logits": d.decode_step(t["tokens"], at, return_logits=True), "k": d.k_cache, "v": d.v_cache}
    return lambda: {"logits": d.prefill(t["tokens"], return_logits=True), "k": d.k_cache, "v": d.v_cache}


def prepare(case, seed):
    t = _weights(case, seed)
    call = {"w4": _linears, "w8": _linears, "mlp": _mlp, "experts": _experts, "fused": _experts, "decode": _stack,
            "prefill": _stack}[case["kind"]](case, t)
    state = {"call": call, "tensors": t}
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # the pass that capture wants before it
            call()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call()
        state.update(graph=graph, out=out)
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ---------------------------------------------------------------- what a pass cannot do without
def _w4_bytes(n, k):
    return n * k // 2 + 4 * n * (k // GROUP)


def work(case):
    kind, m = case["kind"], case["rows"]
    if kind == "w4":
        k, n = case["inp"], case["out"]
        return {"bytes": case["layers"] * (_w4_bytes(n, k) + 2 * m * n) + 2 * m * k, "flops": case["layers"] * 2 * m * n * k}
    if kind == "w8":
        k, n = case["inp"], case["out"]
        return {"bytes": case["layers"] * (n * k + 4 * n + 2 * m * n) + 2 * m * k, "flops": case["layers"] * 2 * m * n * k}
    if kind == "mlp":
        h, i = case["inp"], case["inter"]
        return {"bytes": case["layers"] * (3 * h * i + 8 * i + 6 * h + 6 * m * h) + 2 * m * h, "flops": case["layers"] * 6 * m * h * i}
    if kind in ("experts", "fused"):
        h, i, e, r = case["inp"], case["inter"], case["experts"], case["rows"] * case["top"]
        hit = e * (1.0 - (1.0 - case["top"] / e) ** m)  # experts that get a row, in the mean
        return {"bytes": hit * (3 * h * i + 8 * i + 4 * h) + 4 * m * h + 12 * r, "flops": 6 * r * h * i}
    h, kv, i, v = case["heads"] * HEAD, case["kv"], case["inter"], case["vocab"]
    per = ((case["heads"] + 2 * kv) * HEAD, h), (h, h), (2 * i, h), (h, i)
    weights = case["layers"] * sum(_w4_bytes(*p) for p in per) + _w4_bytes(v, h)
    macs = case["layers"] * sum(n * k for n, k in per)
    if kind == "decode":
        ctx = case["context"] + 1
        return {"bytes": weights + case["layers"] * 4 * m * kv * ctx * HEAD + 2 * m * (h + v),
                "flops": 2 * m * (macs + v * h) + case["layers"] * 4 * m * ctx * h}
    return {"bytes": weights + case["layers"] * 4 * m * kv * HEAD + 2 * m * h + 2 * v,
            "flops": 2 * m * macs + 2 * v * h + case["layers"] * 2 * m * m * h}


def tolerance(case):
    # four times what the paths are off exact(): one product deep that is the output's rounding and the int4 weights' (fp16 2e-4 to
    # 4e-4, bf16 2e-3), and the chains, which requantize in between, show no more; a stack's roundings travel (fp16 1.4e-3)
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 5e-3, "max": 0.1}
    if case["kind"] in ("w4", "w8"):
        return {"rel": 1.5e-3 if case["dtype"] == "fp16" else 8e-3, "max": 0.05}
    return {"rel": 2e-3 if case["dtype"] == "fp16" else 8e-3, "max": 0.1}


# ---------------------------------------------------------------- the same in 64 bits
def _w4_values(w):
    packed, scales, zeros = w
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    u = ((packed.unsqueeze(-1) >> shifts) & 15).flatten(1).double()
    return (u - zeros.double().repeat_interleave(GROUP, 1)) * scales.double().repeat_interleave(GROUP, 1)


def _fake(t):
    """Per-token 8-bit fake quantization in the tensor's own dtype."""
    s = t.abs().amax(-1, keepdim=True).clamp(min=1e-5) / 127
    return (t / s).round() * s


def _dynamic(t):
    """Per-token 8-bit quantization with a 32-bit scale, as values in 64 bits."""
    t = t.float()
    s = t.abs().amax(-1, keepdim=True) / 127
    return (t / s).round().clamp(-128, 127).double() * s.double()


def _values(w, dtype=None):
    """An int8 weight's values; with a dtype, rounded to it as a fake-quantized weight is held."""
    codes, scales = w
    v = codes.float() * scales.unsqueeze(-1)
    return (v if dtype is None else v.to(dtype)).double()


def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w.double()


def _exact_experts(case, t):
    (w13, w2), _ = t["layers"][0]
    fake, dt = case["kind"] == "experts", DTYPES[case["dtype"]]
    x = _fake(t["x"]).double() if fake else _dynamic(t["x"])
    out = torch.zeros_like(x)
    for e in range(case["experts"]):
        tok, slot = torch.where(t["ids"] == e)
        if tok.numel() == 0:
            continue
        gu = x[tok] @ _values((w13[0][e], w13[1][e]), dt if fake else None).T
        if fake:  # the module's tensors are held in its dtype up to the down projection
            g, u = gu.to(dt).chunk(2, -1)
            h = _fake(torch.nn.functional.silu(g) * u).double()
        else:
            g, u = gu.chunk(2, -1)
            h = _dynamic(torch.nn.functional.silu(g) * u)
        out.index_add_(0, tok, (h @ _values((w2[0][e], w2[1][e]), dt if fake else None).T) * t["topw"][tok, slot, None].double())
    return out


def _rope64(x, pos):
    inv = 1.0 / (10000.0 ** (torch.arange(0, HEAD, 2, device="cuda").float() / HEAD))
    f = torch.outer(pos.float(), inv)  # the tables are held in fp16
    cos, sin = f.cos().half().double(), f.sin().half().double()
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _exact_stack(case, t):
    decode, heads, kv, inter = case["kind"] == "decode", case["heads"], case["kv"], case["inter"]
    rows, grp = case["rows"], heads // kv
    x = t["embed"][t["tokens"].reshape(-1)].double()
    ks, vs = [], []
    for li, l in enumerate(t["layers"]):
        qkv = (_rms64(x, l["ln1"]) @ _w4_values(l["qkv"]).T).view(rows, heads + 2 * kv, HEAD).transpose(0, 1)
        q, k, v = qkv[:heads], qkv[heads:heads + kv], qkv[heads + kv:]
        att = torch.empty(rows, heads, HEAD, dtype=torch.float64, device="cuda")
        if decode:
            pos = torch.full((rows,), case["context"], device="cuda")
            kc, vc = t["k"][li].double(), t["v"][li].double()
            kc[:, :, -1], vc[:, :, -1] = _rope64(k, pos).transpose(0, 1), v.transpose(0, 1)
            q = _rope64(q, pos)
            for b in range(rows):
                for j in range(kv):
                    p = torch.softmax(q[j * grp:(j + 1) * grp, b] @ kc[b, j].T / math.sqrt(HEAD), -1)
                    att[b, j * grp:(j + 1) * grp] = p @ vc[b, j]
        else:
            pos = torch.arange(rows, device="cuda")
            q, kc, vc = _rope64(q, pos), _rope64(k, pos), v
            later = torch.ones(rows, rows, device="cuda", dtype=torch.bool).triu(1)
            for j in range(heads):
                s = (q[j] @ kc[j // grp].T / math.sqrt(HEAD)).masked_fill_(later, float("-inf"))
                att[:, j] = torch.softmax(s, -1) @ vc[j // grp]
            kc, vc = kc.unsqueeze(0), vc.unsqueeze(0)
        ks.append(kc)
        vs.append(vc)
        x = x + att.flatten(1) @ _w4_values(l["o"]).T
        gu = _rms64(x, l["ln2"]) @ _w4_values(l["gate_up"]).T
        x = x + (torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]) @ _w4_values(l["down"]).T
    last = x if decode else x[-1:]
    logits = last * torch.rsqrt(last.square().mean(-1, keepdim=True) + 1e-5) @ _w4_values(t["lm_head"]).T
    return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}


@torch.no_grad()
def exact(case, seed):
    t, kind = _weights(case, seed), case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_stack(case, t)
    if kind in ("experts", "fused"):
        return _exact_experts(case, t)
    out = []
    for w, b in t["layers"]:
        if kind == "mlp":
            w13, w2, ln, res = w
            total = t["x"].double() + res.double()  # the norm is of the sum before it is rounded to the residual
            y = _rms64(total, torch.ones_like(ln)).to(ln.dtype) * ln
            g, u = (_dynamic(y) @ _values(w13).T).chunk(2, -1)
            out += [_dynamic(torch.nn.functional.silu(g) * u) @ _values(w2).T, total.to(ln.dtype).double()]
            continue
        if kind == "w4":
            y = t["x"].double() @ _w4_values(w).T
        else:
            y = _fake(t["x"]).double() @ _values(w, t["x"].dtype).T
        out.append(y if b is None else y + b.double())
    return out
