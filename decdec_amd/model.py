"""Decoder-only Transformer whose linear layers are the quantised DEC modules of ``decdec_amd.linear``.

Counterpart of the reference's end-to-end/model.py (a gpt-fast style Llama / Phi-3 decoder): same
``ModelArgs`` fields and model names, fused ``wqkv`` and ``w1w3`` projections, a static KV cache,
``load_dec_data`` / ``create_dec_context`` / ``set_dec_config`` / ``update_dec_config`` with the
reference's meaning (k_chunks = [qkv, o, gate_up, down]).  Everything that is not a linear layer is
plain torch: this file exists to drive the linear-layer hot path from a real decode step, not to be a
model zoo.  A decode step touches only static buffers, so it can be captured in a HIP graph; on the GPU
its residual adds + normalisations, rotary embedding, cache append, attention and gated activation run on the library's
helper kernels
(``decode_ops``), a prefill or CPU pass on torch ops.
"""
from __future__ import annotations

import math
from dataclasses import dataclass
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import decode_ops, ext
from .cache import KVCache, SequenceState
from .linear import may_make, packed_layer, step_layer


def find_multiple(n: int, k: int) -> int:
    return n if n % k == 0 else n + k - n % k


@dataclass
class ModelArgs:
    block_size: int = 2048
    vocab_size: int = 32000
    n_layer: int = 32
    n_head: int = 32
    dim: int = 4096
    intermediate_size: Optional[int] = None
    n_local_heads: int = -1
    head_dim: int = 64
    rope_base: float = 10000
    norm_eps: float = 1e-5
    model_name: Optional[str] = None

    def __post_init__(self):
        if self.n_local_heads == -1:
            self.n_local_heads = self.n_head
        if self.intermediate_size is None:
            self.intermediate_size = find_multiple(int(2 * 4 * self.dim / 3), 256)
        self.head_dim = self.dim // self.n_head

    @classmethod
    def from_name(cls, name: str) -> "ModelArgs":
        if name not in transformer_configs:
            raise KeyError(f"Unknown model name: {name}, available: {sorted(transformer_configs)}")
        return cls(**transformer_configs[name])


# reference end-to-end/model.py:54-58, plus a small shape for tests
transformer_configs = {
    "Meta-Llama-3-8B-Instruct": dict(model_name="Meta-Llama-3-8B-Instruct", block_size=8192, n_layer=32, n_head=32,
                                     n_local_heads=8, dim=4096, intermediate_size=14336, vocab_size=128256,
                                     rope_base=500000),
    "Meta-Llama-3-70B-Instruct": dict(model_name="Meta-Llama-3-70B-Instruct", block_size=8192, n_layer=80, n_head=64,
                                      n_local_heads=8, dim=8192, intermediate_size=28672, vocab_size=128256,
                                      rope_base=500000),
    "Phi-3-medium-4k-instruct": dict(model_name="Phi-3-medium-4k-instruct", block_size=4096, n_layer=40, n_head=40,
                                     n_local_heads=10, dim=5120, intermediate_size=17920, vocab_size=32064,
                                     rope_base=10000),
    "tiny-llama-test": dict(model_name="tiny-llama-test", block_size=256, n_layer=2, n_head=8, n_local_heads=2,
                            dim=512, intermediate_size=1536, vocab_size=640, rope_base=10000),
}


class RMSNorm(nn.Module):
    """x / rms(x) * weight (one fused kernel; statistics in fp32)."""

    def __init__(self, dim: int, eps: float = 1e-5):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return F.rms_norm(x, (x.shape[-1],), self.weight, self.eps)


def rope_frequencies(dims: int, base: float, scaling: Optional[dict] = None):
    """(pair frequencies [dims / 2] in fp64, magnitude of cos and sin).  `scaling` (factor, original, fast, slow) is YaRN's:
    pairs that turn fewer than `slow` times over `original` positions are slowed down by `factor`, pairs that turn more
    than `fast` times are left alone, with a linear ramp over the pair index in between."""
    inv = base ** (-torch.arange(0, dims, 2, dtype=torch.float64) / dims)
    if not scaling:
        return inv, 1.0
    turns_to_dim = lambda t: dims * math.log(scaling["original"] / (2 * math.pi * t)) / (2 * math.log(base))
    lo = max(math.floor(turns_to_dim(scaling["fast"])), 0)
    hi = min(math.ceil(turns_to_dim(scaling["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return inv / scaling["factor"] * ramp + inv * (1 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0


def rope_tables(head_dim: int, max_pos: int, base: float, device=None, layout: str = "half", dims: Optional[int] = None,
                scaling: Optional[dict] = None):
    """cos / sin in fp32.  layout "half": [max_pos, head_dim] for the half-rotation form, pair (i, i + head_dim/2) is
    rotated by pos * base^(-2i/head_dim).  layout "pairs": [max_pos, head_dim / 2], pair (2i, 2i + 1); the first `dims`
    elements (all by default) turn, the rest keep their values; `scaling` as in rope_frequencies."""
    if layout == "half":
        inv_freq = 1.0 / (base ** (torch.arange(0, head_dim, 2, dtype=torch.float32, device=device) / head_dim))
        ang = torch.arange(max_pos, dtype=torch.float32, device=device)[:, None] * inv_freq[None, :]
        ang = torch.cat((ang, ang), dim=-1)
        return ang.cos(), ang.sin()
    dims = head_dim if dims is None else dims
    freq, mag = rope_frequencies(dims, base, scaling)
    ang = torch.arange(max_pos, dtype=torch.float64)[:, None] * freq[None, :]
    cos, sin = torch.ones(max_pos, head_dim // 2), torch.zeros(max_pos, head_dim // 2)
    cos[:, :dims // 2], sin[:, :dims // 2] = (ang.cos() * mag).float(), (ang.sin() * mag).float()
    return cos.to(device), sin.to(device)


def apply_rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """x [..., S, D] with cos / sin [S, D] already gathered at the positions of the S tokens (same dtype)."""
    half = x.shape[-1] // 2
    rot = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos + rot * sin


def neighbours(want, n: int):
    """Places that follow each other among n rows as a slice, None for others.  A list of places as an index is copied from the
    host, and that copy waits for everything the stream was given: 120 us of a short prompt in which nothing new was queued."""
    if type(want) not in (list, tuple, range) or len(want) == 0 or any(type(w) is not int for w in want):
        return None
    first = want[0]
    if not 0 <= first <= n - len(want) or any(w != first + i for i, w in enumerate(want)):
        return None
    return slice(first, first + len(want))


def hooked(m: nn.Module) -> bool:
    """Whether somebody sees the calls of `m`, by a hook of its own or one on all modules."""
    return bool(m._forward_hooks or m._forward_pre_hooks or nn.modules.module._has_any_global_hook())


def _norm_on_kernel(norm, x: torch.Tensor) -> bool:
    """Whether the library's row kernel may take the place of the module `norm` on rows like x: nobody sees its calls."""
    if type(norm) is not RMSNorm or x.shape[-1] % 4 or x.shape[-1] > 16384 or "forward" in norm.__dict__ or hooked(norm):
        return False
    w = norm.weight
    return w.dtype == x.dtype and w.is_contiguous() and w.data_ptr() % 8 == 0 and w.get_device() == x.get_device()


def _read_at_positions(x: torch.Tensor, cos, sin) -> bool:
    """Whether a kernel may read rotary tables itself.  They are attributes: they stay where they are when a model is moved."""
    return ext.plain(x.get_device(), cos, sin) and cos.shape == sin.shape and (cos.data_ptr() | sin.data_ptr()) % 16 == 0


def _add_norm(h: torch.Tensor, y, norm):
    """(h + y, norm of it) of rows that `_norm_on_kernel` holds for; y: None, or what a projection gave, which on the kernel has to be
    like h."""
    if y is not None and (y.dtype != h.dtype or y.shape != h.shape or h.dtype != norm.weight.dtype or y.get_device() != h.get_device()):
        h = h + y
        return h, norm(h)
    if y is not None:
        y = y.contiguous()
        y = y if y.data_ptr() % 8 == 0 else y.clone()
    s, n = h if y is None else torch.empty_like(h), torch.empty_like(h)
    decode_ops.add_rmsnorm(h, y, norm.weight, None if y is None else s, n, norm.eps)
    return s, n


class Attention(nn.Module):
    def __init__(self, config: ModelArgs, linear_class, linear_kwargs):
        super().__init__()
        assert config.dim % config.n_head == 0 and config.n_head % config.n_local_heads == 0
        total = (config.n_head + 2 * config.n_local_heads) * config.head_dim
        self.wqkv = linear_class(config.dim, total, bias=False, **linear_kwargs)
        self.wo = linear_class(config.dim, config.dim, bias=False, **linear_kwargs)
        self.kv_cache: Optional[KVCache] = None
        self.n_head, self.n_local_heads, self.head_dim, self.dim = config.n_head, config.n_local_heads, config.head_dim, config.dim

    def forward(self, x: torch.Tensor, mask: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, input_pos: torch.Tensor,
                rope_tables_full=None, prompt_kernels: bool = False):
        B, S, _ = x.shape
        kv = self.n_local_heads * self.head_dim
        qkv = self.wqkv(x)
        if rope_tables_full is not None and not prompt_kernels:
            return self._step(qkv, input_pos, rope_tables_full)
        if prompt_kernels:
            # several tokens on the library's tiled kernel; `mask` is not needed: a token sees the positions up to its own
            tables = rope_tables_full is not None
            if tables:
                cos, sin = rope_tables_full[:2]
            y = decode_ops.prompt_attention(qkv[0].contiguous(), cos, sin, input_pos, self.kv_cache.k_cache, self.kv_cache.v_cache,
                                            self.n_head, self.n_local_heads, tables)
            return self.wo(y[None])
        # RoPE on the query and key heads in one pass (they are neighbours in the fused projection)
        nqk = self.n_head + self.n_local_heads
        qk = apply_rope(qkv[..., :self.dim + kv].view(B, S, nqk, self.head_dim).transpose(1, 2), cos, sin)
        q, k = qk[:, :self.n_head], qk[:, self.n_head:]
        v = qkv[..., self.dim + kv:].view(B, S, self.n_local_heads, self.head_dim).transpose(1, 2)
        if self.kv_cache is not None:
            k, v = self.kv_cache.update(input_pos, k, v)
        # grouped-query attention over the whole (static) cache; rows of `mask` hide what is not yet written
        y = F.scaled_dot_product_attention(q, k, v, attn_mask=mask, enable_gqa=self.n_head != self.n_local_heads)
        y = y.transpose(1, 2).reshape(B, S, self.dim)
        return self.wo(y)


    def _step(self, qkv, input_pos, rope_tables_full):
        """One token on the library's helper kernel: rotate, append to the cache and attend in one launch."""
        y = torch.empty(1, 1, self.dim, dtype=qkv.dtype, device=qkv.device)
        decode_ops.rope_attention(qkv.view(-1), rope_tables_full[0], rope_tables_full[1], input_pos, y, self.kv_cache.k_cache, self.kv_cache.v_cache, self.n_head,
                                  self.n_local_heads, rope_tables_full[2])
        return self.wo(y)


class FeedForward(nn.Module):
    def __init__(self, config: ModelArgs, linear_class, linear_kwargs):
        super().__init__()
        self.inter = config.intermediate_size
        self.w1w3 = linear_class(config.dim, 2 * self.inter, bias=False, **linear_kwargs)
        self.w2 = linear_class(self.inter, config.dim, bias=False, **linear_kwargs)

    def forward(self, x: torch.Tensor, helper_kernels: bool = False, prompt_kernels: bool = False) -> torch.Tensor:
        gu = self.w1w3(x)
        if prompt_kernels:
            return self.w2(decode_ops.silu_mul_rows(gu[0].contiguous())[None])
        if helper_kernels:
            return self._down(gu)
        a, b = gu.split([self.inter, self.inter], dim=-1)
        return self.w2(F.silu(a) * b)

    def _down(self, gu):
        """One token on the library's helper kernel."""
        act = torch.empty(1, 1, self.inter, dtype=gu.dtype, device=gu.device)
        decode_ops.silu_mul(gu.view(-1), act.view(-1))
        return self.w2(act)


class TransformerBlock(nn.Module):
    def __init__(self, config: ModelArgs, linear_class, linear_kwargs):
        super().__init__()
        self.attention = Attention(config, linear_class, linear_kwargs)
        self.feed_forward = FeedForward(config, linear_class, linear_kwargs)
        self.input_layernorm = RMSNorm(config.dim, config.norm_eps)
        self.post_attention_layernorm = RMSNorm(config.dim, config.norm_eps)

    def forward(self, x, mask, cos, sin, input_pos, rope_tables_full=None, prompt_kernels: bool = False):
        norm = self.post_attention_layernorm
        if prompt_kernels:
            a = self.attention(self.input_layernorm(x), mask, cos, sin, input_pos, prompt_kernels=True)
            if a.dtype == x.dtype and _norm_on_kernel(norm, x):
                # residual and norm in one pass
                h, n = torch.empty_like(x), torch.empty_like(x)
                decode_ops.add_rmsnorm(x, a.contiguous(), norm.weight, h, n, norm.eps)
            else:
                h = x + a
                n = norm(h)
            return h + self.feed_forward(n, prompt_kernels=True)
        h = x + self.attention(self.input_layernorm(x), mask, cos, sin, input_pos, rope_tables_full)
        return h + self.feed_forward(norm(h), rope_tables_full is not None)

    def decode_step(self, h, branch, input_pos, rope_tables_full, normed=None):
        """One token on the helper kernels.  `h` is the residual stream before this block, `branch` the output of
        the previous block's feed-forward that has not been added yet (None for the first block); returns the
        stream after this block's attention and this block's feed-forward output, again not yet added.  `normed`: the first block's norm of
        h, where it is there already."""
        attention, ff, norm1, norm2 = self.attention, self.feed_forward, self.input_layernorm, self.post_attention_layernorm
        makes = self._products_make(h, branch)
        h0 = h if branch is None else torch.empty_like(h)
        if normed is None and makes[0]:
            qkv = decode_ops.norm_product(attention.wqkv, h, branch, norm1.weight, norm1.eps, h0)
            a = attention._step(qkv, input_pos, rope_tables_full)
        else:
            n1 = normed
            if normed is None:
                n1 = torch.empty_like(h)
                decode_ops.add_rmsnorm(h, branch, norm1.weight, None if branch is None else h0, n1, norm1.eps)
            a = attention(n1, None, None, None, input_pos, rope_tables_full)
        h1, at = torch.empty_like(h), h.get_device()
        if makes[1] and a.dtype == h.dtype and a.shape == h.shape and ext.plain(at, a) and a.data_ptr() % 8 == 0:
            gu = decode_ops.norm_product(ff.w1w3, h0, a, norm2.weight, norm2.eps, h1)
        else:
            n2 = torch.empty_like(h)
            decode_ops.add_rmsnorm(h0, a, norm2.weight, h1, n2, norm2.eps)
            if not makes[2]:
                return h1, ff(n2, True)
            gu = ff.w1w3(n2)
        if makes[2] and gu.dtype == h.dtype and gu.numel() == 2 * ff.w2.in_features and ext.plain(at, gu) and gu.data_ptr() % 4 == 0:
            return h1, decode_ops.gate_product(ff.w2, gu.view(-1))
        return h1, ff._down(gu)

    def _products_make(self, h, branch):
        """Whether the queries' product, and that of gate and up, take the norm ahead of them into their launches, and the last one the gate: layers as
        `step_layer` asks for, and nobody sees or changes the calls of the modules in between."""
        attention, ff = self._modules["attention"], self._modules["feed_forward"]
        if type(attention) is not Attention or type(ff) is not FeedForward:
            return False, False, False
        # steps that the host deals out pay for what is asked here: most layers are of another kind
        wqkv, w1w3, w2 = attention._modules["wqkv"], ff._modules["w1w3"], ff._modules["w2"]
        if not (may_make(wqkv) or may_make(w1w3) or may_make(w2)):
            return False, False, False
        norm1, norm2, at, dtype = self._modules["input_layernorm"], self._modules["post_attention_layernorm"], h.get_device(), h.dtype
        if (not ext.on_kernels(h.device, h) or h.data_ptr() % 8
                or (branch is not None and (branch.dtype != dtype or branch.shape != h.shape or not ext.plain(at, branch) or branch.data_ptr() % 8))):
            return False, False, False
        free = [not hooked(m) and "forward" not in m.__dict__ for m in (attention, ff)]
        return (free[0] and "_step" not in attention.__dict__ and step_layer(wqkv, True, dtype, at) and _norm_on_kernel(norm1, h),
                free[1] and "_down" not in ff.__dict__ and step_layer(w1w3, True, dtype, at) and _norm_on_kernel(norm2, h),
                free[1] and ff.inter == getattr(w2, "in_features", 0) and step_layer(w2, False, dtype, at))

    def prompt_step(self, h, branch, input_pos, rope_tables_full):
        """Several tokens, as `decode_step`: `branch` is the previous block's feed-forward, not yet added, and so is the second
        result.  Only where `steps_over` holds."""
        attention, ff = self._modules["attention"], self._modules["feed_forward"]
        layers = self._packed_layers(attention, ff, h, branch)
        if layers is not None:
            # the linear parts in a call each: a short prompt is bound by what the host does for a launch (77 tokens, two blocks, 370 us of calls from here)
            norm1, norm2, rows = self._modules["input_layernorm"], self._modules["post_attention_layernorm"], h.shape[1]
            scratch = torch.empty(decode_ops.prompt_scratch_bytes(rows, h.shape[2], layers[0][4], ff.inter), dtype=torch.uint8, device=h.device)
            qkv, h0 = torch.empty(rows, layers[0][4], dtype=h.dtype, device=h.device), h
            if branch is not None:
                h0 = torch.empty_like(h)
            decode_ops.prompt_front(h, branch, norm1.weight, norm1.eps, layers[0], None if branch is None else h0, qkv, scratch)
            y = decode_ops.prompt_attention(qkv, rope_tables_full[0], rope_tables_full[1], input_pos, attention.kv_cache.k_cache, attention.kv_cache.v_cache,
                                            attention.n_head, attention.n_local_heads, True)
            h1, out = torch.empty_like(h), torch.empty_like(h)
            decode_ops.prompt_back(h0, y, norm2.weight, norm2.eps, layers[1:], h1, out, scratch)
            return h1, out
        h, n = _add_norm(h, branch, self.input_layernorm)
        a = self.attention(n, None, None, None, input_pos, rope_tables_full, prompt_kernels=True)
        h, n = _add_norm(h, a, self.post_attention_layernorm)
        return h, self.feed_forward(n, prompt_kernels=True)

    def _packed_layers(self, attention, ff, h, branch):
        """The four linear layers as `decode_ops.prompt_front` and `prompt_back` take them, None where one of them has to be called by itself."""
        at, dtype, rows, dim = h.get_device(), h.dtype, h.shape[1], h.shape[2]
        if branch is not None and (branch.dtype != dtype or branch.shape != h.shape or not ext.plain(at, branch) or branch.data_ptr() % 8):
            return None
        if not ext.plain(at, h) or h.data_ptr() % 8 or attention.n_head * attention.head_dim != dim:
            return None
        layers, a, f = [], attention._modules, ff._modules
        for l, K, N in ((a["wqkv"], dim, (attention.n_head + 2 * attention.n_local_heads) * attention.head_dim), (a["wo"], dim, dim),
                        (f["w1w3"], dim, 2 * ff.inter), (f["w2"], ff.inter, dim)):
            layer = packed_layer(l, rows, dtype, at)
            if layer is None or layer[3] != K or layer[4] != N:
                return None
            layers.append(layer)
        return layers

    def steps_over(self, x, positions: int) -> bool:
        """Whether nobody sees the calls of this block's parts or changes what they give to `prompt_step`, and the cache has as many
        `positions` as the rotary tables have rows."""
        attention, ff = self._modules["attention"], self._modules["feed_forward"]
        wo, w2 = attention._modules["wo"], ff._modules["w2"]
        if any(m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__ for m in (self, attention, ff, wo, w2)):
            return False
        return (all(getattr(l, "dtype", None) == x.dtype and getattr(l, "out_features", None) == x.shape[-1] for l in (wo, w2))
                and attention.kv_cache.k_cache.shape[2] == positions
                and _norm_on_kernel(self._modules["input_layernorm"], x) and _norm_on_kernel(self._modules["post_attention_layernorm"], x))

    def dec_linears(self):
        """The four compensated linears in the order of the k_chunk lists: qkv, o, gate_up, down."""
        return [self.attention.wqkv, self.attention.wo, self.feed_forward.w1w3, self.feed_forward.w2]


DEC_MODULE_KEYS = ("attention.wqkv", "attention.wo", "feed_forward.w1w3", "feed_forward.w2")


class Transformer(nn.Module):
    def __init__(self, dtype, config: ModelArgs, linear_class=nn.Linear, linear_kwargs=None, device="cuda"):
        super().__init__()
        self.config, self.dtype = config, dtype
        linear_kwargs = dict(linear_kwargs or {})
        self.tok_embeddings = nn.Embedding(config.vocab_size, config.dim, dtype=dtype, device=device)
        self.layers = nn.ModuleList(TransformerBlock(config, linear_class, linear_kwargs) for _ in range(config.n_layer))
        self.norm = RMSNorm(config.dim, config.norm_eps)
        self.output = nn.Linear(config.dim, config.vocab_size, bias=False, dtype=dtype, device=device)
        self.max_batch_size = self.max_seq_length = -1
        self.dec_contexts = []
        # one-token steps use the library's rotary / attention / activation kernels instead of torch ops
        self.decode_kernels = (torch.device(device).type == "cuda" and dtype in (torch.float16, torch.bfloat16)
                               and config.head_dim in (64, 128))
        self.to(device)
        for m in self.modules():
            if isinstance(m, RMSNorm):
                m.weight.data = m.weight.data.to(dtype)

    @classmethod
    def from_name(cls, dtype, name: str, **kw) -> "Transformer":
        return cls(dtype, ModelArgs.from_name(name), **kw)

    def setup_caches(self, max_batch_size: int, max_seq_length: int):
        if self.max_seq_length >= max_seq_length and self.max_batch_size >= max_batch_size:
            return
        max_seq_length = find_multiple(max_seq_length, 8)
        self.max_seq_length, self.max_batch_size = max_seq_length, max_batch_size
        dev = self.tok_embeddings.weight.device
        for b in self.layers:
            b.attention.kv_cache = KVCache(max_batch_size, max_seq_length, self.config.n_local_heads,
                                           self.config.head_dim, self.dtype, dev)
        self.state = SequenceState([b.attention.kv_cache for b in self.layers], max_seq_length)
        self.causal_mask = torch.tril(torch.ones(max_seq_length, max_seq_length, dtype=torch.bool, device=dev))
        cos, sin = rope_tables(self.config.head_dim, max_seq_length, self.config.rope_base, dev)
        self.rope_cos, self.rope_sin = cos.to(self.dtype), sin.to(self.dtype)
        self.attention_workspace = None
        # caches beyond 512 positions: with a workspace the kernel shares a head's positions among up to 8 workgroups
        # once the sequence is longer than that (8.9 against 17.0 us at position 2047; below, one workgroup per head
        # is faster: 5.9 against 8.0 us at 255)
        if self.decode_kernels and max_seq_length > 512:
            self.attention_workspace = decode_ops.attention_workspace(self.config.n_head, self.config.head_dim, dev)

    def share_output_arena(self):
        """Puts the persistent decode outputs of all quantised linears into one buffer that a decode step
        clears with a single fill, instead of one fill per linear."""
        lins = [l for layer in self.layers for l in layer.dec_linears() if hasattr(l, "external_zero")]
        if not lins:
            return
        total = sum(find_multiple(l.out_features, 64) for l in lins)
        self.output_arena = torch.zeros(total, dtype=self.dtype, device=self.tok_embeddings.weight.device)
        off = 0
        for l in lins:
            l.output = self.output_arena[off:off + l.out_features].view(1, 1, l.out_features)
            l.external_zero = True
            off += find_multiple(l.out_features, 64)

    def forward(self, idx: torch.Tensor, input_pos: torch.Tensor, start: Optional[int] = None, want=None) -> torch.Tensor:
        """idx [B, S] token ids, input_pos [S] positions (int64); returns logits [B, S, vocab], or [B, len(want), vocab]
        for the places `want` among the S tokens.  `start` (the first position) is not needed here."""
        assert self.max_seq_length > 0, "Caches must be initialized first"
        assert idx.shape[1] <= self.max_seq_length and input_pos.numel() == idx.shape[1], \
            f"{idx.shape[1]} positions do not fit a cache of {self.max_seq_length} (input_pos must hold one position per token)"
        arena = getattr(self, "output_arena", None) if idx.shape[1] == 1 else None
        if self._opens_on_kernel(idx, arena):
            emb, norm = self.tok_embeddings.weight, self.layers[0].input_layernorm
            h, n = (torch.empty(1, 1, self.config.dim, dtype=emb.dtype, device=emb.device) for _ in range(2))
            if arena is not None:
                ext.written(arena)
            decode_ops.open_step(idx, emb, norm.weight, norm.eps, h, n, arena)
            return self._decode(h, n, input_pos)
        if arena is not None:
            arena.zero_()
        x = self.tok_embeddings(idx)
        if self.decode_kernels and idx.shape == (1, 1) and x.is_cuda:
            return self._decode(x.contiguous(), None, input_pos)
        prompt = self._prompt_on_kernels(x, input_pos)
        rows = None if want is None else neighbours(want, x.shape[1])
        if prompt and len(self.layers) > 0 and (want is None or rows is not None) and _norm_on_kernel(self.norm, x) and x.data_ptr() % 8 == 0 \
                and _read_at_positions(x, self.rope_cos, self.rope_sin) and all(b.steps_over(x, self.rope_cos.shape[0]) for b in self.layers):
            # sums and norms in one pass, and the last ones of the wanted rows alone
            x, branch, full = x.contiguous(), None, (self.rope_cos, self.rope_sin)
            for layer in self.layers:
                x, branch = layer.prompt_step(x, branch, input_pos, full)
            if rows is not None:
                x, branch = x[:, rows].contiguous(), branch.expand_as(x)[:, rows]
            n = _add_norm(x, branch, self.norm)[1]
        else:
            cos, sin = self.rope_cos.index_select(0, input_pos), self.rope_sin.index_select(0, input_pos)
            mask = None if prompt else self.causal_mask.index_select(0, input_pos)      # [S, max_seq]
            for layer in self.layers:
                x = layer(x, mask, cos, sin, input_pos, prompt_kernels=True) if prompt else layer(x, mask, cos, sin, input_pos)
            if want is not None:
                x = x[:, want] if rows is None else x[:, rows]
            n = self.norm(x)
        head = self.output
        if prompt and n.shape[1] == 1 and type(head) is nn.Linear and head.weight.is_contiguous() and head.weight.data_ptr() % 16 == 0 \
                and not hooked(head):
            return self._head_of_one(n.contiguous())
        return self.output(n)

    def _decode(self, h, normed, input_pos):
        """Logits of one token on the helper kernels: h its embedding, normed the first norm of it where it is there."""
        full, branch = (self.rope_cos, self.rope_sin, self.attention_workspace), None
        for layer in self.layers:
            if normed is None:
                h, branch = layer.decode_step(h, branch, input_pos, full)
            else:
                h, branch = layer.decode_step(h, branch, input_pos, full, normed)
                normed = None
        n = torch.empty_like(h)
        decode_ops.add_rmsnorm(h, branch, self.norm.weight, torch.empty_like(h), n, self.norm.eps)
        return self._head_of_one(n)

    def _opens_on_kernel(self, idx, arena) -> bool:
        """Whether one launch may embed the token, take the first block's norm and clear the arena: one token, modules as they are here, nobody sees the
        embedding's call."""
        if not self.decode_kernels or idx.shape != (1, 1) or len(self.layers) == 0 or idx.dtype != torch.int64 or not idx.is_cuda:
            return False
        emb, first = self.tok_embeddings, self.layers[0]
        if type(emb) is not nn.Embedding or emb.max_norm is not None or "forward" in emb.__dict__ or hooked(emb) or type(first) is not TransformerBlock \
                or "decode_step" in first.__dict__:
            return False
        w, norm = emb.weight, first.input_layernorm
        if torch.is_grad_enabled() and (w.requires_grad or norm.weight.requires_grad):
            return False
        tensors = (idx, w, norm.weight) if arena is None else (idx, w, norm.weight, arena)
        if not _norm_on_kernel(norm, w) or not ext.on_kernels(idx.device, *tensors) or w.dtype not in (torch.float16, torch.bfloat16) or w.shape[1] != self.config.dim:
            return False
        return w.data_ptr() % 8 == 0 and (arena is None or (arena.data_ptr() % 16 == 0 and arena.numel() * arena.element_size() % 16 == 0))

    def _head_of_one(self, n: torch.Tensor) -> torch.Tensor:
        """Logits of one token: the unquantised head on the library's streaming GEMV (a gigabyte of weights at 8B)."""
        if self.output.bias is None and self.output.weight.dtype == n.dtype and self.config.dim % 8 == 0:
            logits = torch.empty(1, 1, self.config.vocab_size, dtype=n.dtype, device=n.device)
            decode_ops.dense_gemv(self.output.weight, n.view(-1), logits.view(-1))
            return logits
        return self.output(n)

    def _prompt_on_kernels(self, x: torch.Tensor, input_pos: torch.Tensor) -> bool:
        """Whether the attention of several tokens runs on the library's kernel: one sequence, inference, blocks as they are here,
        nothing that has to see torch operations."""
        if any(type(b) is not TransformerBlock or type(b.attention) is not Attention or type(b.feed_forward) is not FeedForward
               or type(b.attention.kv_cache) is not KVCache for b in self.layers):
            return False
        caches = [t for b in self.layers for t in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache)]
        return (self.decode_kernels and x.shape[0] == 1 and x.shape[1] > 1 and not torch.is_grad_enabled() and not torch.is_autocast_enabled()
                and input_pos.dtype == torch.int64 and input_pos.dim() == 1 and caches[0].shape[0] == 1 and x.dtype == caches[0].dtype
                and ext.on_kernels(x.device, x, input_pos, *caches))

    # ---- DEC plumbing (reference end-to-end/model.py:143-215) ----
    def load_dec_data(self, dec_data: dict):
        for i, layer in enumerate(self.layers):
            for key, lin in zip(DEC_MODULE_KEYS, layer.dec_linears()):
                p = f"layers.{i}.{key}."
                lin.load_dec_data(dec_data[p + "q_residual"], dec_data[p + "scales"], dec_data[p + "thresholds"])

    def create_dec_context(self, n_tbs, buffer_size: int = 1024):
        n_tbs = [n_tbs] if isinstance(n_tbs, int) else list(n_tbs)
        dev = self.tok_embeddings.weight.device
        self.selected_rows_buffers = [torch.empty(buffer_size, dtype=torch.int32, device=dev) for _ in n_tbs]
        self.selected_activations_buffers = [torch.empty(buffer_size, dtype=self.dtype, device=dev) for _ in n_tbs]
        self.dec_contexts = [ext.create_dec_context(n, r, a) for n, r, a in
                             zip(n_tbs, self.selected_rows_buffers, self.selected_activations_buffers)]

    def update_dec_context(self, n_tbs):
        n_tbs = [n_tbs] if isinstance(n_tbs, int) else list(n_tbs)
        assert len(n_tbs) == len(self.dec_contexts)
        old = self.dec_contexts
        self.dec_contexts = [ext.create_dec_context(n, r, a) for n, r, a in
                             zip(n_tbs, self.selected_rows_buffers, self.selected_activations_buffers)]
        self._stale_contexts = getattr(self, "_stale_contexts", []) + old      # configs may still point at them

    def _k_chunks(self, k_chunks):
        k_chunks = list(k_chunks)
        assert len(k_chunks) == 4, "k_chunks = [qkv, o, gate_up, down]"
        return k_chunks

    def set_dec_config(self, k_chunks):
        for layer in self.layers:
            for lin, k in zip(layer.dec_linears(), self._k_chunks(k_chunks)):
                lin.create_dec_config(self.dec_contexts[0], k)

    def update_dec_config(self, k_chunks):
        for layer in self.layers:
            for lin, k in zip(layer.dec_linears(), self._k_chunks(k_chunks)):
                lin.update_dec_config(self.dec_contexts[0], k)
