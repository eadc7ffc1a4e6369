"""The work that users have this framework do, as cases of a size: what is timed, on which inputs, and how exact it is.

Six kinds, each through its public entry point:

linear          one quantised layer at batch 1 (``decdec_amd.linear``), with or without error compensation: the drop-in use
                of the ops, one call at a time, where latency and launches count
token           the linear layers of some decoder layers in one captured graph (``decdec_amd.ext``), q | k | v and
                gate | up in one launch each: the decode-time hot path by itself
decode          one greedy step of a decoder with quantised linears (``generate.DecodeStep``, captured)
prefill         a prompt fed to such a decoder (``generate.Session``): logits of its last token, keys and values of all
hybrid_decode,
hybrid_prefill  the same two for the decoders of checkpoint folders (Fivitar, Fekulix)

Models are cut to a few layers of the named shapes; weights, caches and tokens are random and made from the seed alone.
"""
from __future__ import annotations

import math

import torch

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
# width, feed-forward, query heads, key heads, vocabulary, rotary base, longest sequence
PLAIN = {"Meta-Llama-3-8B-Instruct": (4096, 14336, 32, 8, 128256, 500000.0, 8192),
         "Phi-3-medium-4k-instruct": (5120, 17920, 40, 10, 32064, 10000.0, 4096)}
LLAMA, PHI = PLAIN
HEAD = 128                                             # head size of every model here
HYBRID = {2048: (16, 8, 7168), 4096: (32, 8, 14336)}   # width: heads, key heads, feed-forward
HYBRID_VOCAB, EPS = 32000, 1e-6
GROUP = 128                                            # channels that share a scale (lutgemm)


def listed():
    return [
        # one key projection through the drop-in module: a few microseconds of work, latency and launches are all of it
        {"name": "linear_sqllm4_k", "kind": "linear", "format": "sqllm", "bits": 4, "dtype": "fp16", "K": 4096, "N": 1024, "k_chunk": 0},
        # the longest rows of a medium model, compensated, binary-coded
        {"name": "linear_lutgemm3_down_dec", "kind": "linear", "format": "lutgemm", "bits": 3, "dtype": "bf16", "K": 17920, "N": 5120, "k_chunk": 8},
        # the compensated decode path by itself, residuals in host memory
        {"name": "token_anyprec3_dec", "kind": "token", "layers": 4, "bits": 3, "dtype": "fp16", "k_chunk": 32, "n_tb": 32},
        # a decode step far into a conversation, without compensation
        {"name": "decode_llama_sqllm4", "kind": "decode", "model": LLAMA, "layers": 4, "format": "sqllm", "bits": 4, "dtype": "fp16", "pos": 2000, "k_chunk": 0},
        # a compensated decode step soon after a short prompt
        {"name": "decode_phi_lutgemm3_dec", "kind": "decode", "model": PHI, "layers": 2, "format": "lutgemm", "bits": 3, "dtype": "fp16", "pos": 300, "k_chunk": 4},
        # the prompt of the end-to-end experiment
        {"name": "prefill_llama_sqllm4", "kind": "prefill", "model": LLAMA, "layers": 2, "format": "sqllm", "bits": 4, "dtype": "fp16", "tokens": 512},
        # a long prompt of no particular length
        {"name": "prefill_llama_anyprec3", "kind": "prefill", "model": LLAMA, "layers": 2, "format": "anyprec", "bits": 3, "dtype": "bf16", "tokens": 1999},
        # a chat turn
        {"name": "prefill_phi_lutgemm3", "kind": "prefill", "model": PHI, "layers": 2, "format": "lutgemm", "bits": 3, "dtype": "fp16", "tokens": 77},
        # a long document through the hybrid decoder, all its mixers once
        {"name": "fivitar_prefill", "kind": "hybrid_prefill", "design": "Fivitar", "width": 4096, "layers": 3, "dtype": "bf16", "tokens": 8192, "portion": 4096},
        # its decode step behind that document
        {"name": "fivitar_decode", "kind": "hybrid_decode", "design": "Fivitar", "width": 4096, "layers": 3, "dtype": "bf16", "pos": 8000},
        # a prompt of no particular length with 32-bit storage, the command line's option for checking a checkpoint
        {"name": "fekulix_prefill_fp32", "kind": "hybrid_prefill", "design": "Fekulix", "width": 2048, "layers": 2, "dtype": "fp32", "tokens": 777, "portion": 4096},
        # a decode step of the smaller model
        {"name": "fekulix_decode", "kind": "hybrid_decode", "design": "Fekulix", "width": 2048, "layers": 4, "dtype": "bf16", "pos": 1500},
    ]


def _between(rng, lo, hi):
    """A whole number of lo .. hi, its logarithm spread evenly."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "token", "decode", "decode", "prefill", "prefill", "prefill", "hybrid_decode", "hybrid_prefill", "hybrid_prefill"])
    fmt, bits = rng.choice([("sqllm", 4), ("sqllm", 3), ("anyprec", 3), ("anyprec", 4), ("lutgemm", 3), ("lutgemm", 4)])
    dt16 = rng.choice(["fp16", "bf16"])
    if kind == "linear":
        step = GROUP if fmt == "lutgemm" else 32
        return {"kind": kind, "format": fmt, "bits": bits, "dtype": dt16, "K": max(1, _between(rng, 512, 17920) // step) * step,
                "N": _between(rng, 256, 35840) // 8 * 8, "k_chunk": rng.choice([0, 0, 4, 8, 16, 32])}
    if kind == "token":
        return {"kind": kind, "layers": rng.randint(1, 3), "bits": rng.choice([3, 4]), "dtype": dt16, "k_chunk": rng.choice([0, 4, 8, 16, 32]), "n_tb": rng.choice([16, 32])}
    model = {"model": rng.choice([LLAMA, PHI]), "layers": rng.randint(1, 2), "format": fmt, "bits": bits, "dtype": dt16}
    if kind == "decode":
        return {"kind": kind, **model, "pos": _between(rng, 16, 3800), "k_chunk": rng.choice([0, 0, 4, 8])}
    if kind == "prefill":
        return {"kind": kind, **model, "layers": 1, "tokens": _between(rng, 2, 3000)}
    width, dt = rng.choice([2048, 4096]), rng.choice(["bf16", "bf16", "bf16", "fp32"])
    model = {"design": rng.choice(["Fivitar", "Fekulix"]), "width": width, "layers": rng.randint(2, 3), "dtype": dt}
    if kind == "hybrid_decode":
        return {"kind": kind, **model, "pos": _between(rng, 16, 16000)}
    return {"kind": kind, **model, "tokens": _between(rng, 8, 8192 if dt == "bf16" else 800), "portion": rng.choice([256, 4096, 8192])}


# ---- inputs: everything from the seed, by plain torch on the GPU -----------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000 + seed)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _words(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, generator=g, device="cuda", dtype=torch.int32)


def _quantised(g, fmt, bits, dtype, K, N, std=0.02):
    """The tensors of one quantised layer by the buffer's name: random indices, weights of about `std`."""
    if fmt == "lutgemm":
        step = 5.0 * std / (2 ** bits - 1)
        alpha = (0.75 + 0.5 * torch.rand(K // GROUP, 1, N, generator=g, device="cuda")) * step / 2 * (2.0 ** torch.arange(bits, device="cuda")).view(1, -1, 1)
        return {"qweight": _words(g, K // 32, bits, N), "alpha": alpha.to(dtype), "q_bias": (_randn(g, K // GROUP, N) * std * 0.05).to(dtype)}
    q = _words(g, bits, N, K // 32) if fmt == "anyprec" else _words(g, K * bits // 32, N)
    return {"qweight": q, "lut": (_randn(g, N, 2 ** bits).sort(1).values * std).to(dtype)}


def _activation(g, K, dtype):
    """N(0, 1) with one channel in a hundred twenty times as large."""
    x = _randn(g, K)
    return torch.where(torch.rand(K, generator=g, device="cuda") < 0.01, 20 * x, x).to(dtype)


def _thresholds(samples):
    """[K] on the host: the largest i-th largest magnitude over calibration vectors [draws, K]."""
    return samples.abs().sort(1, descending=True).values.amax(0).cpu()


def _residual(g, K, N, dtype):
    """4-bit residual words and the scales in the ops' order, both on the host."""
    return _words(g, K, N // 8).cpu(), ((torch.rand(N, generator=g, device="cuda") + 0.5) * 2e-4).to(dtype).cpu()


def _llama_linears():
    return [("q", 4096, 4096), ("k", 4096, 1024), ("v", 4096, 1024), ("o", 4096, 4096), ("gate", 4096, 14336), ("up", 4096, 14336), ("down", 14336, 4096)]


def _linear_inputs(case, seed):
    g, dtype, K, N = _gen(seed), DTYPES[case["dtype"]], case["K"], case["N"]
    d = {"w": _quantised(g, case["format"], case["bits"], dtype, K, N), "x": _activation(g, K, dtype)}
    if case["k_chunk"]:
        d["th"] = _thresholds(torch.stack([_activation(g, K, dtype) for _ in range(16)]))
        d["res"], d["scales"] = _residual(g, K, N, dtype)
    return d


def _token_inputs(case, seed):
    g, dtype = _gen(seed), DTYPES[case["dtype"]]
    side = {}
    if case["k_chunk"]:
        for K in (4096, 14336):
            side[K] = _thresholds(torch.stack([_activation(g, K, dtype) for _ in range(16)]))
        for _, K, N in _llama_linears():              # layers of one shape have the same residual words (in memory of their own)
            if (K, N) not in side:
                side[K, N] = _residual(g, K, N, dtype)
    layers = []
    for _ in range(case["layers"]):
        xs = {"q": _activation(g, 4096, dtype), "o": _activation(g, 4096, dtype), "gate": _activation(g, 4096, dtype), "down": _activation(g, 14336, dtype)}
        xs.update(k=xs["q"], v=xs["q"], up=xs["gate"])
        layers.append([{"name": n, "K": K, "N": N, "x": xs[n], "w": _quantised(g, "anyprec", case["bits"], dtype, K, N)} for n, K, N in _llama_linears()])
    return layers, side


LINEARS = ("attention.wqkv", "attention.wo", "feed_forward.w1w3", "feed_forward.w2")


def _plain_shapes(case):
    dim, ff, heads, kv, vocab, base, longest = PLAIN[case["model"]]
    return dict(zip(LINEARS, [(dim, (heads + 2 * kv) * HEAD), (dim, dim), (dim, 2 * ff), (ff, dim)]))


def _plain_weights(case, seed):
    g, dtype = _gen(seed), DTYPES[case["dtype"]]
    dim, ff, heads, kv, vocab, base, longest = PLAIN[case["model"]]
    norm = lambda: (1 + 0.1 * _randn(g, dim)).to(dtype)
    w = {"embed": _randn(g, vocab, dim).to(dtype), "head": (_randn(g, vocab, dim) * 0.02).to(dtype), "norm": norm(), "layers": []}
    for _ in range(case["layers"]):
        layer = {n: _quantised(g, case["format"], case["bits"], dtype, K, N) for n, (K, N) in _plain_shapes(case).items()}
        layer.update(norm1=norm(), norm2=norm())
        w["layers"].append(layer)
    if case.get("k_chunk"):
        # calibration vectors of the sublayers' inputs: normed; an average of values; gated
        std = 0.02 * dim ** 0.5
        kinds = {"attention.wqkv": _randn(g, 8, dim), "attention.wo": _randn(g, 8, dim) * 3 * std / case["pos"] ** 0.5,
                 "feed_forward.w1w3": _randn(g, 8, dim), "feed_forward.w2": _silu(_randn(g, 8, ff) * std) * _randn(g, 8, ff) * std}
        w["dec"] = {n: (*_residual(g, K, N, dtype), _thresholds(kinds[n].to(dtype))) for n, (K, N) in _plain_shapes(case).items()}
    w["gen"] = g
    return w


def _plain_caches(case, w):
    """Keys and values [1, key heads, pos, head size] of the tokens before a decode step, by layer."""
    dim, _, _, kv, *_ = PLAIN[case["model"]]
    make = lambda: (_randn(w["gen"], 1, kv, case["pos"], HEAD) * 0.02 * dim ** 0.5).to(DTYPES[case["dtype"]])
    return [(make(), make()) for _ in range(case["layers"])]


def _tokens(case, seed, vocab):
    n = case.get("tokens", 1)
    return torch.randint(0, vocab, (n,), generator=torch.Generator(device="cuda").manual_seed(7000 + seed), device="cuda")


def _hybrid_config(case):
    heads, kv, ff = HYBRID[case["width"]]
    if case["design"] == "Fivitar":
        yarn = {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}
        kinds = [("lightning", {"heads": heads, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-2 - 6 * i / heads) for i in range(heads)]}),
                 ("delta", {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4}),
                 ("latent_attention", {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
                                       "rot": {"base": 10000.0, "dims": 64, "scaling": yarn}})]
    else:
        kinds = [("parallel", {"left": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": {"base": 10000.0, "dims": 64}},
                               "right": {"heads": heads // 2, "dim": 128, "vdim": 128, "tau": 16.0}, "left_scale": 0.7, "right_scale": 0.6}),
                 ("channel_delta", {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4})]
    return {"architecture": case["design"], "vocab": HYBRID_VOCAB, "width": case["width"], "norm": {"eps": EPS}, "logit_scale": 1.0,
            "layers": [{"type": kinds[i % len(kinds)][0], "mixer": kinds[i % len(kinds)][1], "mlp": {"kind": "dense", "ff": ff}} for i in range(case["layers"])]}


def _mixer_shapes(kind, m, d, rank=128):
    if kind == "parallel":
        return {f"{side}.{n}": s for side, k in (("left", "grouped"), ("right", "gated_linear")) for n, s in _mixer_shapes(k, m[side], d).items()}
    H, D, V = m["heads"], m["dim"], m["vdim"]
    if kind == "grouped":
        G = m["kv_heads"]
        return {"q": (H * D, d), "k": (G * D, d), "v": (G * V, d), "o": (d, H * V), "q.norm": (D,), "k.norm": (D,), "g": (H, d)}
    if kind == "gated_linear":
        return {"q": (H * D, d), "k": (H * D, d), "v": (H * V, d), "g": (H * V, d), "o": (d, H * V), "norm": (V,), "a1": (rank, d), "a2": (H * D, rank), "a2.b": (H * D,)}
    if kind == "latent_attention":
        R, C = m["rot_dim"], m["kv_rank"]
        return {"q": (H * (D + R), d), "dkv": (C + R, d), "dkv.norm": (C,), "uk": (H * D, C), "uv": (H * V, C), "sink": (H,), "o": (d, H * V)}
    if kind == "lightning":
        return {"q": (H * D, d), "k": (H * D, d), "v": (H * V, d), "g": (H * V, d), "norm": (H * V,), "o": (d, H * V)}
    G, n = m["kv_heads"], m["conv"]
    s = {"q": (G * D, d), "q.conv": (G * D, n), "k": (G * D, d), "k.conv": (G * D, n), "v": (H * V, d), "v.conv": (H * V, n), "b": (H, d), "A_log": (H,), "norm": (V,), "o": (d, H * V)}
    if kind == "channel_delta":
        s.update({"a1": (rank, d), "a2": (H * D, rank), "dt_bias": (H * D,), "g1": (rank, d), "g2": (H * V, rank)})
    else:
        s.update({"a": (H, d), "dt_bias": (H,), "g": (H * V, d)})
    return s


def _hybrid_shapes(cfg):
    d, fekulix = cfg["width"], cfg["architecture"] == "Fekulix"
    norm = lambda n: {n: (d,), n + ".b": (d,), n + ".alpha": ()} if fekulix else {n: (d,)}
    out = {"embed": (cfg["vocab"], d), "head": (cfg["vocab"], d), **norm("final.norm")}
    for i, l in enumerate(cfg["layers"]):
        ff = l["mlp"]["ff"]
        s = {"mix." + n: sh for n, sh in _mixer_shapes(l["type"], l["mixer"], d).items()}
        s.update({**norm("norm1"), **norm("norm2"), "mlp.up": (ff, d), "mlp.down": (d, ff)})
        if not fekulix:
            s.update({"rg1": (d, d), "rg1.b": (d,), "rg2": (d, d), "rg2.b": (d,), "mlp.act": (2,)})
        out.update({f"l{i}.{n}": sh for n, sh in s.items()})
    return out


def _hybrid_weights(case, seed):
    g, w = _gen(seed), {}
    for name, shape in _hybrid_shapes(_hybrid_config(case)).items():
        t = _randn(g, *shape)
        if name.endswith(("A_log", "dt_bias")):
            t = t - 2.0                                # from channels that forget soon to ones that keep for thousands of tokens
        elif name.endswith("sink"):
            t = t + 1.0
        elif name.endswith("alpha"):
            t = 0.6 + 0.1 * t
        elif "norm" in name and name.endswith(".b"):
            t = 0.3 * t
        elif "norm" in name:
            t = 1.0 + 0.1 * t
        elif name.endswith(".conv"):
            t = 0.5 * t
        elif len(shape) == 2 and name != "embed":
            t = t / shape[1] ** 0.5
        w[name] = t.to(DTYPES[case["dtype"]])
    return w, g


def _hybrid_past(case, g):
    """What the tokens before a decode step left behind, by layer and mixer, in the layout of the framework's caches."""
    dtype, pos, past = DTYPES[case["dtype"]], case["pos"], []
    for l in _hybrid_config(case)["layers"]:
        m, kind = l["mixer"], l["type"]
        p = {}
        if kind == "latent_attention":
            p["rows"] = _randn(g, pos, m["kv_rank"] + m["rot_dim"]).to(dtype)
        elif kind == "parallel":
            a, b = m["left"], m["right"]
            p["keys"], p["values"] = _randn(g, a["kv_heads"], pos, a["dim"]).to(dtype), _randn(g, a["kv_heads"] * a["vdim"], pos).to(dtype)
            p["state"] = 3 * _randn(g, b["heads"], b["dim"], b["vdim"])
        else:
            p["state"] = (2.0 if kind == "lightning" else 0.3) * _randn(g, m["heads"], m["dim"], m["vdim"])
            if "conv" in m:
                p["ring"] = _randn(g, m["conv"], (2 * m["kv_heads"] * m["dim"] + m["heads"] * m["vdim"])).to(dtype)
        past.append(p)
    return past


# ---- the passes -----------------------------------------------------------------------------------------------------------
class _State:
    """What a user's program holds; handles are given back with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        from decdec_amd import ext
        for c in getattr(self, "configs", []):
            ext.destroy_dec_config(c)
        for c in getattr(self, "contexts", []):
            ext.destroy_dec_context(c)


def _context(n_tb, size, dtype):
    from decdec_amd import ext
    rows, acts = torch.zeros(size, dtype=torch.int32, device="cuda"), torch.zeros(size, dtype=dtype, device="cuda")
    return ext.create_dec_context(n_tb, rows, acts)


def _module(case, fmt, K, N):
    from decdec_amd import linear
    dtype = DTYPES[case["dtype"]]
    if fmt == "lutgemm":
        return linear.LUTGEMMLinear(K, N, case["bits"], GROUP, dtype=dtype)
    return (linear.APLinear if fmt == "anyprec" else linear.SQLLMLinear)(K, N, case["bits"], dtype=dtype)


def _fill(module, tensors):
    for name, t in tensors.items():
        getattr(module, name).copy_(t)


def _prepare_linear(case, seed):
    d = _linear_inputs(case, seed)
    K, N, dtype = case["K"], case["N"], DTYPES[case["dtype"]]
    lin = _module(case, case["format"], K, N)
    _fill(lin, d["w"])
    s = _State(kind="linear", linear=lin, x=d["x"].view(1, 1, K))
    if case["k_chunk"]:
        s.contexts = [_context(16, K, dtype)]
        lin.load_dec_data(d["res"], d["scales"], d["th"])
        lin.create_dec_config(s.contexts[0], case["k_chunk"])
        s.configs = [lin.dec_config]
    return s


def _prepare_token(case, seed):
    from decdec_amd import ext
    layers, side = _token_inputs(case, seed)
    dtype, kc = DTYPES[case["dtype"]], case["k_chunk"]
    s = _State(kind="token", contexts=[], configs=[])
    outs = [torch.zeros(1, 1, l["N"], dtype=dtype, device="cuda") for layer in layers for l in layer]
    # one buffer for all outputs: a step clears it with a single fill
    arena = torch.zeros(sum(t.numel() for t in outs), dtype=dtype, device="cuda")
    at, views = 0, []
    for t in outs:
        views.append(arena[at:at + t.numel()].view(1, 1, -1))
        at += t.numel()
    flat = [l for layer in layers for l in layer]
    if kc:
        s.contexts = [_context(case["n_tb"], 14336, dtype) for _ in range(3)]      # layers of one launch have a context each
        which = {"q": 0, "k": 1, "v": 2, "o": 0, "gate": 0, "up": 1, "down": 0}
        s.configs = [ext.create_dec_config(s.contexts[which[l["name"]]], kc, side[l["K"], l["N"]][0], side[l["K"], l["N"]][1], side[l["K"]]) for l in flat]
    cfgs = s.configs if kc else [0] * len(flat)

    def step():
        arena.zero_()
        for b in range(0, len(flat), 7):
            for group in ([0, 1, 2], [3], [4, 5], [6]):
                ids = [b + i for i in group]
                ext.dec_anyprec_batch([cfgs[i] for i in ids], flat[ids[0]]["x"].view(1, 1, -1), [views[i] for i in ids], [flat[i]["w"]["qweight"] for i in ids],
                                      [flat[i]["w"]["lut"] for i in ids], case["bits"])
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.synchronize()
    s.graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s.graph, stream=stream):
        step()
    s.layers, s.side, s.views = layers, side, views
    return s


def _plain_model(case, seed):
    from decdec_amd import linear
    from decdec_amd.model import ModelArgs, Transformer
    w = _plain_weights(case, seed)
    args = ModelArgs.from_name(case["model"])
    args.n_layer = case["layers"]
    cls = {"sqllm": linear.SQLLMLinear, "anyprec": linear.APLinear, "lutgemm": linear.LUTGEMMLinear}[case["format"]]
    kw = {"bitwidth": case["bits"], "dtype": DTYPES[case["dtype"]]}
    if case["format"] == "lutgemm":
        kw["group_size"] = GROUP
    m = Transformer(DTYPES[case["dtype"]], args, linear_class=cls, linear_kwargs=kw)
    with torch.no_grad():
        m.tok_embeddings.weight.copy_(w["embed"])
        m.output.weight.copy_(w["head"])
        m.norm.weight.copy_(w["norm"])
        for layer, lw in zip(m.layers, w["layers"]):
            layer.input_layernorm.weight.copy_(lw["norm1"])
            layer.post_attention_layernorm.weight.copy_(lw["norm2"])
            for name, lin in zip(LINEARS, layer.dec_linears()):
                _fill(lin, lw[name])
    m.share_output_arena()
    return m.eval(), w


def _prepare_decode(case, seed):
    from decdec_amd.generate import DecodeStep
    m, w = _plain_model(case, seed)
    pos = case["pos"]
    m.setup_caches(1, min(PLAIN[case["model"]][6], pos + 128))
    s = _State(kind="decode", model=m, pos=pos)
    if case["k_chunk"]:
        m.load_dec_data({f"layers.{i}.{n}.{k}": t for i in range(case["layers"]) for n, d in w["dec"].items() for k, t in zip(("q_residual", "scales", "thresholds"), d)})
        m.create_dec_context(16, buffer_size=max(K for K, _ in _plain_shapes(case).values()))
        m.set_dec_config([case["k_chunk"]] * 4)
        s.contexts, s.configs = list(m.dec_contexts), [lin.dec_config for layer in m.layers for lin in layer.dec_linears()]
    for e, (k, v) in zip(m.state.entries, _plain_caches(case, w)):
        e.k_cache[:, :, :pos] = k
        e.v_cache[:, :, :pos] = v
    s.token = int(_tokens(case, seed, PLAIN[case["model"]][4])[0])
    s.step = DecodeStep(m, 64, keep_logits=True)
    s.step.start(s.token, pos)
    s.step.capture()
    return s


def _prepare_prefill(case, seed):
    m, _ = _plain_model(case, seed)
    n = case["tokens"]
    return _State(kind="prefill", model=m, tokens=_tokens(case, seed, PLAIN[case["model"]][4]), portion=4096,
                  room=min(PLAIN[case["model"]][6], n + 256))


def _hybrid_model(case, seed):
    from decdec_amd import registry
    cfg = _hybrid_config(case)
    w, g = _hybrid_weights(case, seed)
    m = registry.model_class(cfg).from_config(cfg, DTYPES[case["dtype"]])
    m.load_weights(w)
    return m.eval(), g


def _prepare_hybrid_prefill(case, seed):
    m, _ = _hybrid_model(case, seed)
    return _State(kind="hybrid_prefill", model=m, tokens=_tokens(case, seed, HYBRID_VOCAB), portion=case["portion"], room=case["tokens"] + 256)


def _parts(entry):
    return entry.parts if hasattr(entry, "parts") else [entry]


def _prepare_hybrid_decode(case, seed):
    from decdec_amd.generate import DecodeStep
    m, g = _hybrid_model(case, seed)
    pos = case["pos"]
    m.setup_caches(1, pos + 128)
    for e, p in zip(m.state.entries, _hybrid_past(case, g)):
        for part in _parts(e):
            if hasattr(part, "rows"):
                part.rows[:pos] = p["rows"]
            elif hasattr(part, "keys"):
                part.keys[:, :pos], part.values[:, :pos] = p["keys"], p["values"]
            else:
                part.state.copy_(p["state"])
                if part.ring is not None:
                    part.ring.copy_(p["ring"])
    s = _State(kind="hybrid_decode", model=m, pos=pos, token=int(_tokens(case, seed, HYBRID_VOCAB)[0]))
    s.held = [t for e in m.state.entries for t in e.recurrent()]
    s.saved = [t.clone() for t in s.held]
    s.step = DecodeStep(m, 64, keep_logits=True)
    s.step.start(s.token, pos)
    s.step.capture()
    return s


PREPARE = {"linear": _prepare_linear, "token": _prepare_token, "decode": _prepare_decode, "prefill": _prepare_prefill,
           "hybrid_decode": _prepare_hybrid_decode, "hybrid_prefill": _prepare_hybrid_prefill}


def prepare(case, seed):
    with torch.no_grad():
        return PREPARE[case["kind"]](case, seed)


def _left_behind(entry, lo, hi):
    """What tokens lo .. hi - 1 changed of a sequence's state."""
    out = {}
    for part in _parts(entry):
        if hasattr(part, "k_cache"):
            out.update(k=part.k_cache[:, :, lo:hi], v=part.v_cache[:, :, lo:hi])
        elif hasattr(part, "rows"):
            out.update(rows=part.rows[lo:hi])
        elif hasattr(part, "keys"):
            out.update(keys=part.keys[:, lo:hi], values=part.values[:, lo:hi])
        else:
            out.update(state=part.state)
            if part.ring is not None:
                out.update(ring=part.ring)
    return out


def run(s):
    if s.kind == "linear":
        return s.linear(s.x)
    if s.kind == "token":
        s.graph.replay()
        return s.views
    if s.kind.endswith("decode"):
        if getattr(s, "saved", None):                  # every pass is the same step: the recurrent layers go back to before it
            torch._foreach_copy_(s.held, s.saved)
        s.step.start(s.token, s.pos)
        s.step.run(1)
        # the token itself may flip between logits that are almost equal: its logit says the same and does not
        return {"logits": s.step.logits, "picked": s.step.logits.gather(1, s.step.token), "state": [_left_behind(e, s.pos, s.pos + 1) for e in s.model.state.entries]}
    from decdec_amd.generate import Session
    n = s.tokens.numel()
    session = Session(s.model, s.room, portion=s.portion)
    logits = session.feed(s.tokens, [n - 1])
    session.close()
    return {"logits": logits, "state": [_left_behind(e, 0, n) for e in s.model.state.entries]}


# ---- the least work -------------------------------------------------------------------------------------------------------
def _packed_bytes(fmt, bits, K, N):
    if fmt == "lutgemm":
        return K * N * bits / 8 + K // GROUP * (bits + 1) * N * 2
    return K * N * bits / 8 + N * 2 ** bits * 2


def work(case):
    kind, size = case["kind"], 4 if case["dtype"] == "fp32" else 2
    if kind == "linear":
        K, N = case["K"], case["N"]
        rows = case["k_chunk"] * K // 1024
        return {"bytes": _packed_bytes(case["format"], case["bits"], K, N) + rows * N / 2 + 2 * (K + N), "flops": 2 * (K + rows) * N}
    if kind == "token":
        by = fl = 0
        for _, K, N in _llama_linears():
            rows = case["k_chunk"] * K // 1024
            by += case["layers"] * (_packed_bytes("anyprec", case["bits"], K, N) + rows * N / 2 + 2 * (K + N))
            fl += case["layers"] * 2 * (K + rows) * N
        return {"bytes": by, "flops": fl}
    rows = case.get("tokens", 1)
    seen = rows if "tokens" in case else case["pos"] + 1      # keys
    pairs = rows * (rows + 1) / 2 if "tokens" in case else seen
    if kind in ("decode", "prefill"):
        dim, ff, heads, kv, vocab, _, _ = PLAIN[case["model"]]
        by, fl = size * (vocab * dim + rows * dim + vocab), 2 * vocab * dim
        for K, N in _plain_shapes(case).values():
            extra = case.get("k_chunk", 0) * K // 1024
            by += case["layers"] * (_packed_bytes(case["format"], case["bits"], K, N) + extra * N / 2)
            fl += case["layers"] * 2 * rows * (K + extra) * N
        by += case["layers"] * 2 * seen * kv * HEAD * size
        fl += case["layers"] * 4 * pairs * heads * HEAD
        return {"bytes": by, "flops": fl}
    cfg = _hybrid_config(case)
    by, fl = size * rows * case["width"], 0
    for name, shape in _hybrid_shapes(cfg).items():
        if name != "embed":
            by += math.prod(shape) * size
        if len(shape) == 2 and name not in ("embed", "head") and not name.endswith(".conv"):
            fl += 2 * rows * math.prod(shape)
    fl += 2 * HYBRID_VOCAB * case["width"]
    for l in cfg["layers"]:
        m = l["mixer"]
        for part in ([m["left"], m["right"]] if l["type"] == "parallel" else [m]):
            H, D, V = part["heads"], part["dim"], part["vdim"]
            if "kv_rank" in part:
                by += seen * (part["kv_rank"] + part["rot_dim"]) * size
                fl += 2 * pairs * H * (D + part["rot_dim"] + V)
            elif "rot" in part:
                by += seen * part["kv_heads"] * (D + V) * size
                fl += 2 * pairs * H * (D + V)
            else:
                by += 2 * H * D * V * 4
                fl += 4 * rows * H * D * V
    return {"bytes": by, "flops": fl}


def tolerance(case):
    # Largest relative errors seen against 64 bits, times about four (and never over what two 16-bit storages may differ by):
    # one layer rounds its output a few times, a model's every sublayer rounds its activations.
    bf16 = case["dtype"] == "bf16"
    if case["kind"] in ("linear", "token"):
        return {"rel": 0.02 if bf16 else 0.002, "max": 0.2 if bf16 else 0.02}
    if case["dtype"] == "fp32":
        return {"rel": 1e-4, "max": 1e-2}
    return {"rel": 0.03 if bf16 else 0.012, "max": 0.9 if bf16 else 0.4}


# ---- 64 bits --------------------------------------------------------------------------------------------------------------
def _sigmoid(z):
    return 1 / (1 + torch.exp(-z))


def _silu(z):
    return z * _sigmoid(z)


def _softplus(z):
    return torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs()))


def _rms(x, weight, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight


def _bits(words, n):
    """The n lowest bits of int32 words, in a new last dimension."""
    return (words[..., None] >> torch.arange(n, device=words.device, dtype=torch.int32)) & 1


def _dense(w, fmt, bits):
    """The weight [N, K] of a quantised layer."""
    q = w["qweight"]
    if fmt == "lutgemm":
        KT, _, N = q.shape
        out = w["q_bias"].double().repeat_interleave(GROUP, 0)                              # [K, N]
        for p in range(bits):
            sign = _bits(q[:, p], 32).permute(0, 2, 1).reshape(KT * 32, N).double() * 2 - 1
            out += sign * w["alpha"][:, p].double().repeat_interleave(GROUP, 0)
        return out.t()
    if fmt == "sqllm":
        N = q.shape[1]
        flat = _bits(q.t().contiguous(), 32).reshape(N, -1, bits)                           # one little-endian stream per output
        idx = (flat << torch.arange(bits, device=q.device, dtype=torch.int32)).sum(-1)
    else:
        _, N, W = q.shape
        K = W * 32
        word, bit = torch.arange(W, device=q.device)[:, None], torch.arange(32, device=q.device)[None, :]
        chunk, t = word // 32, word % 32
        wide = torch.where(chunk == K // 1024, K % 1024 // 32, 32)
        channel = 1024 * chunk + 8 * wide * ((31 - bit) // 8) + 8 * t + (31 - bit) % 8      # of a bit of a word
        idx = torch.zeros(N, K, dtype=torch.int64, device=q.device)
        acc = sum(_bits(q[p], 32).long() << (bits - 1 - p) for p in range(bits))
        idx[:, channel.reshape(-1)] = acc.reshape(N, K)
    return torch.gather(w["lut"].double(), 1, idx.long())


def _selected(x, th, k_chunk):
    """Channels that are compensated: in every 1024, the first k_chunk by magnitude class, then by number.  Class borders
    are computed in the activations' own arithmetic."""
    K, dtype = x.numel(), x.dtype
    to = lambda v: v.to(dtype).float()
    a, b = th[0].float().cpu(), th[k_chunk * K // 1024 - 1].float().cpu()
    i = torch.arange(16, dtype=torch.float32)
    low = to(a + to(to(b - a) * i / 15))
    floors = torch.cat([low, to(b * (15 - i) / 16)]).to(x.device)
    mag, out = x.float().abs(), []
    for lo in range(0, K, 1024):
        seg = mag[lo:lo + 1024]
        cls = (floors[None, :] > seg[:, None]).sum(1)
        out.append(lo + torch.sort(cls, stable=True).indices[:k_chunk * seg.numel() // 1024])
    return torch.cat(out)


def _compensation(x, res, scales, th, k_chunk):
    rows = _selected(x, th, k_chunk)
    words = res.to(x.device)[rows]
    nib = (words[..., None] >> (4 * torch.arange(8, device=x.device, dtype=torch.int32))) & 15          # [k, N / 8, 8]
    scale = scales.to(x.device).double().view(8, -1).t().reshape(-1)
    return (x[rows].double() @ (nib - 8).double().view(rows.numel(), -1)) * scale


def _exact_linear(case, seed):
    d = _linear_inputs(case, seed)
    y = _dense(d["w"], case["format"], case["bits"]) @ d["x"].double()
    if case["k_chunk"]:
        y += _compensation(d["x"], d["res"], d["scales"], d["th"], case["k_chunk"])
    return y.view(1, 1, -1)


def _exact_token(case, seed):
    layers, side = _token_inputs(case, seed)
    out = []
    for layer in layers:
        for l in layer:
            y = _dense(l["w"], "anyprec", case["bits"]) @ l["x"].double()
            if case["k_chunk"]:
                y += _compensation(l["x"], *side[l["K"], l["N"]], side[l["K"]], case["k_chunk"])
            out.append(y.view(1, 1, -1))
    return out


def _attend(q, k, v, start, scale, sink=None):
    """q [H, T, D] on k [G, S, D], v [G, S, V], query i sees keys 0 .. start + i; sink [H]: a score without a value."""
    H, T, _ = q.shape
    G, S, _ = k.shape
    out = torch.empty(T, H, v.shape[-1], dtype=q.dtype, device=q.device)
    hidden = torch.arange(S, device=q.device)[None, :] > start + torch.arange(T, device=q.device)[:, None]
    for h in range(H):
        s = (q[h] @ k[h // (H // G)].t() * scale).masked_fill(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(T, 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :S] @ v[h // (H // G)]
    return out


def _exact_plain(case, seed):
    w = _plain_weights(case, seed)
    dim, ff, heads, kv, vocab, base, _ = PLAIN[case["model"]]
    kc, decode = case.get("k_chunk", 0), case["kind"] == "decode"
    start = case["pos"] if decode else 0
    past = _plain_caches(case, w) if decode else None
    tokens = _tokens(case, seed, vocab)
    T = tokens.numel()
    x = w["embed"][tokens].double()
    ang = (start + torch.arange(T, device="cuda", dtype=torch.float64))[:, None] * base ** (-torch.arange(0, HEAD, 2, device="cuda", dtype=torch.float64) / HEAD)
    cos, sin = torch.cat([ang, ang], 1).cos(), torch.cat([ang, ang], 1).sin()
    turn = lambda t: t * cos + torch.cat([-t[..., HEAD // 2:], t[..., :HEAD // 2]], -1) * sin
    dtype, state = DTYPES[case["dtype"]], []

    def linear(layer, name, h):
        y = h @ _dense(layer[name], case["format"], case["bits"]).t()
        if kc:
            y += _compensation(h[0].to(dtype), *w["dec"][name], kc)
        return y
    for i, layer in enumerate(w["layers"]):
        qkv = linear(layer, "attention.wqkv", _rms(x, layer["norm1"].double(), 1e-5)).view(T, -1, HEAD).transpose(0, 1)
        q, k, v = turn(qkv[:heads]), turn(qkv[heads:heads + kv]), qkv[heads + kv:]
        state.append({"k": k[None], "v": v[None]})
        if decode:
            k, v = torch.cat([past[i][0][0].double(), k], 1), torch.cat([past[i][1][0].double(), v], 1)
        x = x + linear(layer, "attention.wo", _attend(q, k, v, start, HEAD ** -0.5).reshape(T, -1))
        gu = linear(layer, "feed_forward.w1w3", _rms(x, layer["norm2"].double(), 1e-5))
        x = x + linear(layer, "feed_forward.w2", _silu(gu[:, :ff]) * gu[:, ff:])
    logits = _rms(x[-1:], w["norm"].double(), 1e-5) @ w["head"].double().t()
    return {"logits": logits, "picked": logits.max().view(1, 1), "state": state} if decode else {"logits": logits, "state": state}


def _turned(x, start, rot):
    """x [..., T, n]: pairs (2i, 2i + 1) of the first rot["dims"] elements turned by position x frequency (YaRN's scaling)."""
    dims, s = rot["dims"], rot.get("scaling")
    f, mag = rot["base"] ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=x.device) / dims), 1.0
    if s:
        at = lambda turns: dims * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))
        lo, hi = max(math.floor(at(s["fast"])), 0), min(math.ceil(at(s["slow"])), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=torch.float64, device=x.device) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f, mag = f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1.0
    ang = (start + torch.arange(x.shape[-2], dtype=torch.float64, device=x.device))[:, None] * f
    c, n = ang.cos() * mag, ang.sin() * mag
    a, b, y = x[..., 0:dims:2], x[..., 1:dims:2], x.clone()
    y[..., 0:dims:2], y[..., 1:dims:2] = a * c - b * n, b * c + a * n
    return y


def _walk(q, k, v, decay, beta, S):
    """A state [H, D, V] taken through the tokens: decayed (by [T, H, 1 or D, 1]), then k u^T added; u is v, or with beta
    [T, H] the delta rule's beta (v - S^T k).  Read-outs [T, H, V]."""
    out = torch.empty(v.shape, dtype=v.dtype, device=v.device)
    for t in range(q.shape[0]):
        S = S * decay[t]
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], S)[:, 0])
        S = torch.baddbmm(S, k[t][:, :, None], u[:, None])
        out[t] = torch.bmm(q[t][:, None], S)[:, 0]
    return out, S


def _exact_mixer(kind, m, w, h, start, past, left):
    """Read-out behind the output projection; `left` receives what the tokens leave behind."""
    T = h.shape[0]
    if kind == "parallel":
        part = lambda side: {n[len(side) + 1:]: t for n, t in w.items() if n.startswith(side + ".")}
        a = _exact_mixer("grouped", m["left"], part("left"), h, start, past, left)
        b = _exact_mixer("gated_linear", m["right"], part("right"), h, start, past, left)
        return m["left_scale"] * a + m["right_scale"] * b
    H, D, V = m["heads"], m["dim"], m["vdim"]
    if kind == "latent_attention":
        R, C = m["rot_dim"], m["kv_rank"]
        q = (h @ w["q"].t()).view(T, H, D + R).transpose(0, 1)
        q = torch.cat([q[..., :D], _turned(q[..., D:], start, m["rot"])], -1)
        down = h @ w["dkv"].t()
        rows = torch.cat([_rms(down[:, :C], w["dkv.norm"], EPS), _turned(down[:, C:], start, m["rot"])], 1)
        left["rows"] = rows
        if past:
            rows = torch.cat([past["rows"].double(), rows])
        k = (rows[:, :C] @ w["uk"].t()).view(-1, H, D).transpose(0, 1)
        k = torch.cat([k, rows[:, C:].expand(H, -1, R)], -1)
        v = (rows[:, :C] @ w["uv"].t()).view(-1, H, V).transpose(0, 1)
        return _attend(q, k, v, start, m["scale"], w["sink"]).reshape(T, -1) @ w["o"].t()
    if kind == "grouped":
        G = m["kv_heads"]
        q, k, v = ((h @ w[n].t()).view(T, g, -1) for n, g in (("q", H), ("k", G), ("v", G)))
        q = _turned(_rms(q, w["q.norm"], EPS).transpose(0, 1), start, m["rot"])
        k = _turned(_rms(k, w["k.norm"], EPS).transpose(0, 1), start, m["rot"])
        v = v.transpose(0, 1)
        left["keys"], left["values"] = k, v.transpose(1, 2).reshape(G * V, T)
        if past:
            k = torch.cat([past["keys"].double(), k], 1)
            v = torch.cat([past["values"].double().view(G, V, -1).transpose(1, 2), v], 1)
        o = _attend(q, k, v, start, m["scale"], torch.zeros(H, dtype=h.dtype, device=h.device))
        return (o * _sigmoid(h @ w["g"].t())[:, :, None]).reshape(T, -1) @ w["o"].t()
    S = past["state"].double() if past else torch.zeros(H, D, V, dtype=h.dtype, device=h.device)
    beta = None
    if kind in ("delta", "channel_delta"):
        G, n = m["kv_heads"], m["conv"]
        raw = torch.cat([h @ w[c].t() for c in "qkv"], 1)
        before = torch.stack([past["ring"][(start - b) % n] for b in range(n - 1, 0, -1)]).double() if past else raw.new_zeros(n - 1, raw.shape[1])
        ext, taps = torch.cat([before, raw]), torch.cat([w[c + ".conv"] for c in "qkv"])
        ring = past["ring"].double() if past else raw.new_zeros(n, raw.shape[1])
        for t in range(max(0, T - n), T):
            ring[(start + t) % n] = raw[t]
        left["ring"] = ring
        y = _silu(sum(taps[:, j] * ext[j:j + T] for j in range(n)))
        q, k, v = y[:, :G * D].view(T, G, D), y[:, G * D:2 * G * D].view(T, G, D), y[:, 2 * G * D:].view(T, H, V)
        unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
        q, k = (unit(q) * D ** -0.5).repeat_interleave(H // G, 1), unit(k).repeat_interleave(H // G, 1)
        beta = _sigmoid(h @ w["b"].t())
        if kind == "delta":
            decay = torch.exp(-torch.exp(w["A_log"]) * _softplus(h @ w["a"].t() + w["dt_bias"]))[:, :, None, None]
            gate = _silu(h @ w["g"].t())
        else:
            decay = torch.exp(-torch.exp(w["A_log"])[:, None] * _softplus(h @ w["a1"].t() @ w["a2"].t() + w["dt_bias"]).view(T, H, D))[..., None]
            gate = _sigmoid(h @ w["g1"].t() @ w["g2"].t())
    else:
        q, k, v = ((h @ w[n].t()).view(T, H, -1) for n in "qkv")
        if kind == "lightning":
            q, k, v = _silu(q), _silu(k), _silu(v)
            decay = torch.tensor(m["decay"], dtype=h.dtype, device=h.device)[:, None, None].expand(T, H, 1, 1)
            gate = _sigmoid(h @ w["g"].t())
        else:
            q = q * D ** -0.5
            decay = torch.exp(-_softplus(-(h @ w["a1"].t() @ w["a2"].t() + w["a2.b"])) / m["tau"]).view(T, H, D, 1)
            gate = _silu(h @ w["g"].t())
    o, left["state"] = _walk(q, k, v, decay, beta, S)
    o = _rms(o.reshape(T, -1), w["norm"], EPS) if kind == "lightning" else _rms(o, w["norm"], EPS).reshape(T, -1)
    return (o * gate) @ w["o"].t()


def _exact_hybrid(case, seed):
    cfg, decode = _hybrid_config(case), case["kind"] == "hybrid_decode"
    weights, g = _hybrid_weights(case, seed)
    past = _hybrid_past(case, g) if decode else [None] * case["layers"]
    start = case["pos"] if decode else 0
    x = weights["embed"][_tokens(case, seed, HYBRID_VOCAB)].double()
    tanh = lambda x, w, n: torch.tanh(w[n + ".alpha"] * x) * w[n] + w[n + ".b"]
    state = []
    for i, l in enumerate(cfg["layers"]):
        w = {n[len(f"l{i}."):]: t.double() for n, t in weights.items() if n.startswith(f"l{i}.")}
        mix = {n[4:]: t for n, t in w.items() if n.startswith("mix.")}
        left = {}
        if case["design"] == "Fivitar":
            y = _exact_mixer(l["type"], l["mixer"], mix, x, start, past[i], left)
            x = x + _rms(y * _sigmoid(x @ w["rg1"].t() + w["rg1.b"]), w["norm1"], EPS)
            z = x @ w["mlp.up"].t()
            neg, (p, q) = torch.clamp(z, max=0), _softplus(w["mlp.act"])
            act = torch.where(z > 0, p * z * z + z / 2, (0.5 + q) * (torch.exp(neg) - 1 - neg) + neg / 2)
            x = x + _rms(act @ w["mlp.down"].t() * _sigmoid(x @ w["rg2"].t() + w["rg2.b"]), w["norm2"], EPS)
        else:
            x = x + _exact_mixer(l["type"], l["mixer"], mix, tanh(x, w, "norm1"), start, past[i], left)
            z = tanh(x, w, "norm2") @ w["mlp.up"].t()
            x = x + (z / 2 * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))) @ w["mlp.down"].t()
        state.append(left)
    w = {n: weights[n].double() for n in weights if n.startswith("final")}
    x = _rms(x[-1:], w["final.norm"], EPS) if case["design"] == "Fivitar" else tanh(x[-1:], w, "final.norm")
    logits = x @ weights["head"].double().t()
    return {"logits": logits, "picked": logits.max().view(1, 1), "state": state} if decode else {"logits": logits, "state": state}


EXACT = {"linear": _exact_linear, "token": _exact_token, "decode": _exact_plain, "prefill": _exact_plain,
         "hybrid_decode": _exact_hybrid, "hybrid_prefill": _exact_hybrid}


def exact(case, seed):
    with torch.no_grad():
        return EXACT[case["kind"]](case, seed)
