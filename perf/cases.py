"""The work that programs built on this package do, as cases that can be timed and compared.

A case is one of four kinds of call:

  linear    one eager ``ops.int4_linear`` on ``m`` rows, with or without bias.
  layers    the seven linears of ``layers`` decoder layers on ``m`` rows, called as a decoder calls
            them: q, k, v together, o, gate and up together, down.  ``graph``: captured in a HIP
            graph and replayed, as serving loops run batched decode; otherwise eager, as prefill
            is run.  ``concat``: q|k|v and gate|up are one weight each (``int4_linear``), as
            ``fuse_decoder_linears_`` lays them out; otherwise they are siblings
            (``int4_linear_grouped``), as ``group_sibling_linears_`` calls them.
  model     one greedy decode step of the package's TinyLlama-architecture model up to its logits,
            captured in a HIP graph (the fused launches: RMSNorm, RoPE and cache, SwiGLU, residual).
  quantize  ``ops.int4_quantize`` of the seven weights of a decoder layer, as loading a model does.

Layer shapes are those of the package's benchmark (TinyLlama and Qwen2.5-1.5B) and a generic layer
of hidden size 4096.  Weights are N(0, 0.02^2) and activations N(0, 1), as in the benchmark.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "kernel-forge_amd"))

from kernelforge import ops, tinyllama  # noqa: E402

DEV = "cuda"
_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}

TINYLLAMA = {"hidden": 2048, "kv": 256, "inter": 5632}
QWEN = {"hidden": 1536, "kv": 256, "inter": 8960}
LARGE = {"hidden": 4096, "kv": 1024, "inter": 14336}  # a generic layer

# Every drawn case stays below the work of the largest listed one (prefill_m517_large).
_MAX_MACS = 517 * 218_103_808


def listed() -> list[dict]:
    return [
        # The smallest call: one k or v projection of one token, eagerly.  Launch and host latency.
        {"name": "linear_m1", "kind": "linear", "m": 1, "n": 256, "k": 2048, "group": 128, "bias": False},
        # A small batch through a layer with an odd number of rows, fine groups and a bias.
        {"name": "linear_m6_ragged", "kind": "linear", "m": 6, "n": 1001, "k": 6144, "group": 64, "bias": True},
        # Single-stream decode: the linears of the benchmark's model, one token.
        {"name": "decode_m1", "kind": "layers", "m": 1, **TINYLLAMA, "group": 128, "layers": 6, "graph": True,
         "concat": False},
        # The whole decode step of the package's own model.
        {"name": "decode_model", "kind": "model", "group": 128, "layers": 22, "max_seq": 160, "pos": 77},
        # Small decode batches, the second model, fine groups.
        {"name": "batch_m4_g64", "kind": "layers", "m": 4, **QWEN, "group": 64, "layers": 6, "graph": True,
         "concat": False},
        # Batched decode at the usual batch sizes of a server, odd ones among them.
        {"name": "batch_m16", "kind": "layers", "m": 16, **TINYLLAMA, "group": 128, "layers": 6, "graph": True,
         "concat": False},
        {"name": "batch_m27_large", "kind": "layers", "m": 27, **LARGE, "group": 128, "layers": 1, "graph": True,
         "concat": False},
        {"name": "batch_m64", "kind": "layers", "m": 64, **TINYLLAMA, "group": 128, "layers": 6, "graph": True,
         "concat": True},
        {"name": "batch_m200", "kind": "layers", "m": 200, **QWEN, "group": 128, "layers": 6, "graph": True,
         "concat": False},
        # Prefill of an odd-length prompt through a large layer, and the benchmark's 2,048 tokens.
        {"name": "prefill_m517_large", "kind": "layers", "m": 517, **LARGE, "group": 128, "layers": 1, "graph": False,
         "concat": True},
        {"name": "prefill_m2048", "kind": "layers", "m": 2048, **TINYLLAMA, "group": 128, "layers": 1, "graph": False,
         "concat": False},
        # Loading a model: a layer's bf16 weights into the packed format.
        {"name": "quantize_layer", "kind": "quantize", **TINYLLAMA, "group": 128, "dtype": "bf16"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dims(rng, group: int) -> dict:
    """Layer sizes of the listed models, or any others between them: hidden and inter multiples of
    the group size, kv a multiple of 64."""
    if rng.random() < 0.4:
        return dict(rng.choice([TINYLLAMA, QWEN, LARGE]))
    hidden = group * max(1, round(_log_int(rng, 1024, 4096) / group))
    inter = group * max(1, round(hidden * rng.uniform(2.0, 4.0) / group))
    return {"hidden": hidden, "kv": 64 * rng.randint(2, max(2, hidden // 256)), "inter": inter}


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "layers", "layers", "layers", "model", "quantize"])
    group = rng.choice([64, 128])
    if kind == "linear":
        m = _log_int(rng, 1, 2048)
        k = group * max(1, round(_log_int(rng, 512, 14336) / group))
        n = _log_int(rng, 256, 14336)
        if m > 7 or rng.random() < 0.5:  # above 7 rows the package takes whole multiples of 64
            n = max(64, n // 64 * 64)
        return {"kind": kind, "m": m, "n": n, "k": k, "group": group, "bias": rng.random() < 0.5}
    if kind == "model":
        max_seq = rng.choice([96, 160, 288])
        return {"kind": kind, "group": group, "layers": rng.randint(4, 22), "max_seq": max_seq,
                "pos": rng.randint(1, max_seq - 2)}
    dims = _dims(rng, group)
    if kind == "quantize":
        return {"kind": kind, **dims, "group": group, "dtype": rng.choice(sorted(_DTYPES))}
    params = sum(n * k for _, n, k in _linears(dims))
    graph = rng.random() < 0.7
    m = _log_int(rng, 1, 512) if graph else _log_int(rng, 256, 4096)
    m = min(m, _MAX_MACS // params)
    layers = max(1, min(6, 240_000_000 // params)) if graph else 1
    layers = max(1, min(layers, _MAX_MACS // (params * m)))
    return {"kind": kind, "m": m, **dims, "group": group, "layers": layers, "graph": graph,
            "concat": rng.random() < 0.5}


def _linears(c: dict) -> list[tuple[str, int, int]]:
    """(name, N, K) of a decoder layer's linears."""
    h, kv, i = c["hidden"], c["kv"], c["inter"]
    return [("q", h, h), ("k", kv, h), ("v", kv, h), ("o", h, h), ("gate", i, h), ("up", i, h), ("down", h, i)]


def _calls(c: dict) -> list[list[tuple[int, int]]]:
    """The calls of one decoder layer, each a list of (N, K) weights that share an input."""
    d = {name: (n, k) for name, n, k in _linears(c)}
    calls = [["q", "k", "v"], ["o"], ["gate", "up"], ["down"]]
    if not c["concat"]:
        return [[d[x] for x in names] for names in calls]
    return [[(sum(d[x][0] for x in names), d[names[0]][1])] for names in calls]


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _weight(n: int, k: int, g: torch.Generator, dtype=torch.float32) -> torch.Tensor:
    return (torch.randn(n, k, generator=g, device=DEV) * 0.02).to(dtype)


def _rows(m: int, k: int, g: torch.Generator) -> torch.Tensor:
    return torch.randn(m, k, generator=g, device=DEV).half()


def _capture(fn):
    """fn's calls in a HIP graph, and the outputs that each replay writes."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _run_layers(state) -> list[torch.Tensor]:
    g, ys = state["case"]["group"], []
    for x, ws in state["calls"]:
        if len(ws) == 1:
            ys.append(ops.int4_linear(x, ws[0][0], ws[0][1], g))
        else:
            ys += ops.int4_linear_grouped([x] * len(ws), [w[0] for w in ws], [w[1] for w in ws], g)
    return ys


def prepare(case: dict, seed: int) -> dict:
    gen, kind, s = _gen(seed), case["kind"], {"case": case}
    if kind == "linear":
        s["w"] = ops.int4_quantize(_weight(case["n"], case["k"], gen), case["group"])
        s["x"] = _rows(case["m"], case["k"], gen)
        s["bias"] = torch.randn(case["n"], generator=gen, device=DEV).half() if case["bias"] else None
    elif kind == "layers":
        s["calls"] = [(_rows(case["m"], ns[0][1], gen),
                       [ops.int4_quantize(_weight(n, k, gen), case["group"]) for n, k in ns])
                      for _ in range(case["layers"]) for ns in _calls(case)]
        if case["graph"]:
            s["graph"], s["out"] = _capture(lambda: _run_layers(s))
    elif kind == "model":
        cfg = tinyllama.TinyLlamaConfig(layers=case["layers"], max_seq=case["max_seq"])
        model = tinyllama.build_int4_model(cfg, DEV, seed, case["group"])
        dec = tinyllama.GraphDecoder(model, DEV)
        # The state that a prompt of `pos` tokens leaves: a filled cache, the mask opened up to it.
        dec.cache[:, 0].view(cfg.layers, cfg.kv_heads, cfg.head_dim, cfg.max_seq)[..., :case["pos"]] = torch.randn(
            cfg.layers, cfg.kv_heads, cfg.head_dim, case["pos"], generator=gen, device=DEV).half()
        dec.cache[:, 1, :, :case["pos"]] = torch.randn(cfg.layers, cfg.kv_heads, case["pos"], cfg.head_dim,
                                                       generator=gen, device=DEV).half()
        dec.token.copy_(torch.randint(cfg.vocab, (1,), generator=gen, device=DEV))
        dec.pos.fill_(case["pos"])
        dec.mask[:, :case["pos"] + 1] = 0.0
        s["model"], s["dec"] = model, dec

        def step():
            return model(dec.token, dec.pos, dec.cache, dec.rope, dec.mask, logits_fp32=False)

        s["graph"], logits = _capture(step)
        s["out"] = {"logits": logits, "cache": dec.cache}
    else:
        s["weights"] = [_weight(n, k, gen, _DTYPES[case["dtype"]]) for _, n, k in _linears(case)]
    return s


def run(state):
    case = state["case"]
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if case["kind"] == "linear":
        return ops.int4_linear(state["x"], *state["w"], case["group"], state["bias"])
    if case["kind"] == "layers":
        return _run_layers(state)
    return [ops.int4_quantize(w, case["group"]) for w in state["weights"]]


def _linear_work(m: int, n: int, k: int, group: int) -> tuple[float, float]:
    """(bytes, flops) of one linear without its input rows."""
    return n * k / 2 + 2 * n * k / group + 2 * m * n, 2.0 * m * n * k


def work(case: dict) -> dict:
    g, kind = case["group"], case["kind"]
    if kind == "linear":
        b, f = _linear_work(case["m"], case["n"], case["k"], g)
        return {"bytes": b + 2 * case["m"] * case["k"] + (2 * case["n"] if case["bias"] else 0), "flops": f}
    if kind == "layers":
        b = f = 0.0
        for ns in _calls(case):
            b += 2 * case["m"] * ns[0][1]
            for n, k in ns:
                lb, lf = _linear_work(case["m"], n, k, g)
                b, f = b + lb, f + lf
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    if kind == "model":
        c = tinyllama.TinyLlamaConfig(layers=case["layers"], max_seq=case["max_seq"])
        per = [_linear_work(1, n, k, g) for _, n, k in _linears(TINYLLAMA)]
        # Weights, the cache entries up to the position, the lm_head, one embedding row, the logits.
        kv = 2 * c.kv_heads * c.head_dim * (case["pos"] + 1) * 2
        return {"bytes": c.layers * (sum(b for b, _ in per) + kv) + 2 * c.vocab * (c.hidden + 1) + 2 * c.hidden,
                "flops": c.layers * (sum(f for _, f in per) + 4.0 * c.heads * c.head_dim * (case["pos"] + 1))
                + 2.0 * c.vocab * c.hidden}
    el = 4 if case["dtype"] == "fp32" else 2
    return {"bytes": sum(n * k * (el + 0.5 + 2 / g) for _, n, k in _linears(case)), "flops": 0}


def tolerance(case: dict):
    if case["kind"] == "quantize":
        return "exact"
    # fp16 results of fp32 sums over weights that may or may not be rounded to fp16 first: 2e-4 to
    # 3e-4 of the result against 64 bits.  The model's layers carry such roundings on.
    return {"rel": 6e-3} if case["kind"] == "model" else {"rel": 1.2e-3}


# ---- the same results in 64 bits, in plain torch ----------------------------------------------
_NIBBLE_OF_K = (0, 4, 1, 5, 2, 6, 3, 7)  # nibble position of k offset 0..7 in a packed word


def _dequant64(packed: torch.Tensor, scales: torch.Tensor, group: int) -> torch.Tensor:
    q = torch.stack([((packed >> (4 * p)) & 15) for p in _NIBBLE_OF_K], dim=-1).flatten(1) - 8
    return q.double() * scales.double().repeat_interleave(group, dim=1)


def _linear64(x: torch.Tensor, w, group: int) -> torch.Tensor:
    return x.double() @ _dequant64(w[0], w[1], group).t().contiguous()


def _norm64(x, norm):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + norm.eps) * norm.weight.double()


def _model64(s) -> dict:
    model, dec, case = s["model"], s["dec"], s["case"]
    c, p, g = model.cfg, case["pos"], case["group"]
    d, half = c.head_dim, c.head_dim // 2
    cos, sin = (t[p].double() for t in dec.rope)  # sin carries the sign of rotate-half
    cache = dec.cache.double()
    x = model.embed_tokens.weight[dec.token].double()
    for i, layer in enumerate(model.layers):
        a, m = layer.self_attn, layer.mlp
        qkv = _linear64(_norm64(x, layer.input_layernorm), (a.qkv.packed, a.qkv.scales), g)
        qkv = qkv.view(c.heads + 2 * c.kv_heads, d)
        qk, v = qkv[:c.heads + c.kv_heads], qkv[c.heads + c.kv_heads:]
        qk = qk * cos + torch.cat([qk[:, half:], qk[:, :half]], dim=-1) * sin
        keys = cache[i, 0].view(c.kv_heads, d, c.max_seq)
        keys[..., p], cache[i, 1, :, p] = qk[c.heads:], v
        q = qk[:c.heads].view(c.kv_heads, -1, d)
        probs = torch.softmax(q @ keys[..., :p + 1].contiguous() / math.sqrt(d), dim=-1)
        out = (probs @ cache[i, 1, :, :p + 1].contiguous()).reshape(1, -1)
        x = x + _linear64(out, (a.o_proj.packed, a.o_proj.scales), g)
        gu = _linear64(_norm64(x, layer.post_attention_layernorm), (m.gate_up.packed, m.gate_up.scales), g)
        gate, up = gu.chunk(2, dim=-1)
        x = x + _linear64(torch.nn.functional.silu(gate) * up, (m.down_proj.packed, m.down_proj.scales), g)
    logits = _norm64(x, model.norm) @ model.lm_head.weight.double().t().contiguous()
    return {"logits": logits.view(-1), "cache": cache}


def exact(case: dict, seed: int):
    # Seeds, weights and packing are those of prepare(); only the path's own results are redone.
    s = prepare({**case, "graph": False} if case["kind"] == "layers" else case, seed)
    g = case["group"]
    if case["kind"] == "linear":
        y = _linear64(s["x"], s["w"], g)
        return y if s["bias"] is None else y + s["bias"].double()
    if case["kind"] == "layers":
        return [_linear64(x, w, g) for x, ws in s["calls"] for w in ws]
    if case["kind"] == "model":
        return _model64(s)
    # Quantize: the packed words are whole numbers compared bit for bit; scales are absmax / 7.
    return [(None, (w.double().abs().view(w.shape[0], -1, g).amax(-1) / 7)) for w in s["weights"]]
