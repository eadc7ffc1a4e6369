"""Decode-step helpers of the library (rotary embedding + KV-cache append, one-token grouped-query
attention, gated activation) as functions on torch tensors.  They raise if the HIP library is missing;
there is no fallback."""
from __future__ import annotations

import array
import functools

import torch

from . import _lib
from .ext import _DT, _check, _dt, _ptr, _stream


def _half_cuda(*ts):
    at, dtype = ts[0].get_device(), ts[0].dtype          # -1 on the host
    if at >= 0 and (dtype is torch.float16 or dtype is torch.bfloat16):
        for t in ts:
            if t.get_device() != at or t.dtype is not dtype or not t.is_contiguous():
                break
        else:
            return
    for t in ts:
        _check(at >= 0 and t.get_device() == at and t.is_contiguous(), "tensors must be contiguous CUDA tensors of one GPU")
        _check(t.dtype == ts[0].dtype and t.dtype in (torch.float16, torch.bfloat16), "tensors must share an fp16 / bf16 dtype")


def _pos(pos, beside):
    _check(pos.get_device() == beside.get_device() and pos.dtype == torch.int64 and pos.numel() == 1, "pos must be one int64 on the device")


def _floats(workspace, beside):
    _check(workspace.get_device() == beside.get_device() and workspace.is_contiguous() and workspace.dtype == torch.float32,
           "workspace must be a contiguous float32 CUDA tensor")


def rope_cache_update(qkv: torch.Tensor, cos_table: torch.Tensor, sin_table: torch.Tensor, pos: torch.Tensor,
                      q_out: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, n_head: int, n_kv_head: int) -> None:
    """qkv [(n_head + 2 n_kv_head) * D]; tables [max_seq, D]; pos int64 [1] on the device; caches [1, n_kv_head, max_seq, D]."""
    _half_cuda(qkv, cos_table, sin_table, q_out, k_cache, v_cache)
    _pos(pos, qkv)
    D, max_seq = k_cache.shape[-1], k_cache.shape[-2]
    _check(qkv.numel() == (n_head + 2 * n_kv_head) * D and q_out.numel() == n_head * D, "qkv / q_out size mismatch")
    _check(k_cache.numel() == n_kv_head * max_seq * D and v_cache.shape == k_cache.shape, "cache shape mismatch")
    _check(tuple(cos_table.shape) == (max_seq, D) and tuple(sin_table.shape) == (max_seq, D), "rotary tables must be [max_seq, head_dim]")
    _lib.check(_lib.load().decdec_rope_cache_update(_ptr(qkv), _ptr(cos_table), _ptr(sin_table), _ptr(pos), _ptr(q_out),
                                                    _ptr(k_cache), _ptr(v_cache), _dt(qkv), n_head, n_kv_head, D, max_seq, _stream()))


def attention_workspace(n_head: int, head_dim: int, device="cuda") -> torch.Tensor:
    """Workspace that lets `decode_attention` / `rope_attention` share the positions of a head among up to 8
    workgroups.  It must be zero when first used (it starts with the heads' arrival counters, which every call leaves
    at zero)."""
    n = _lib.load().decdec_decode_attention_workspace_bytes(n_head, head_dim, 8)
    return torch.zeros(n // 4, dtype=torch.float32, device=device)


def decode_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, pos: torch.Tensor,
                     out: torch.Tensor, n_head: int, n_kv_head: int, workspace: torch.Tensor | None = None) -> None:
    _half_cuda(q, k_cache, v_cache, out)
    _pos(pos, q)
    D, max_seq = k_cache.shape[-1], k_cache.shape[-2]
    _check(q.numel() == n_head * D and out.numel() == n_head * D, "q / out size mismatch")
    _check(k_cache.numel() == n_kv_head * max_seq * D and v_cache.shape == k_cache.shape, "cache shape mismatch")
    if workspace is not None:
        _floats(workspace, q)
    _lib.check(_lib.load().decdec_decode_attention(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(pos), _ptr(out), _dt(q),
                                                   n_head, n_kv_head, D, max_seq,
                                                   _ptr(workspace) if workspace is not None else None,
                                                   workspace.numel() * 4 if workspace is not None else 0, _stream()))


def decode_attention_static(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, pos: torch.Tensor,
                            out: torch.Tensor, n_head: int, n_kv_head: int) -> None:
    """`decode_attention` with the library's own static workspace: nothing is allocated and no workspace is passed
    (at most 128 heads; calls on one GPU must not overlap in time)."""
    _half_cuda(q, k_cache, v_cache, out)
    _pos(pos, q)
    D, max_seq = k_cache.shape[-1], k_cache.shape[-2]
    _check(q.numel() == n_head * D and out.numel() == n_head * D, "q / out size mismatch")
    _check(k_cache.numel() == n_kv_head * max_seq * D and v_cache.shape == k_cache.shape, "cache shape mismatch")
    _lib.check(_lib.load().decdec_decode_attention_static(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(pos), _ptr(out),
                                                          _dt(q), n_head, n_kv_head, D, max_seq, _stream()))


def rope_attention(qkv: torch.Tensor, cos_table: torch.Tensor, sin_table: torch.Tensor, pos: torch.Tensor,
                   out: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, n_head: int, n_kv_head: int,
                   workspace: torch.Tensor | None = None) -> None:
    """`rope_cache_update` + `decode_attention` in one launch: un-rotated qkv in, attention output out, the new key /
    value row appended to the caches."""
    _half_cuda(qkv, cos_table, sin_table, out, k_cache, v_cache)
    _pos(pos, qkv)
    D, max_seq = k_cache.shape[-1], k_cache.shape[-2]
    _check(qkv.numel() == (n_head + 2 * n_kv_head) * D and out.numel() == n_head * D, "qkv / out size mismatch")
    _check(k_cache.numel() == n_kv_head * max_seq * D and v_cache.shape == k_cache.shape, "cache shape mismatch")
    _check(tuple(cos_table.shape) == (max_seq, D) and tuple(sin_table.shape) == (max_seq, D), "rotary tables must be [max_seq, head_dim]")
    if workspace is not None:
        _floats(workspace, qkv)
    _lib.check(_lib.linears.decdec_rope_attention(_ptr(qkv), _ptr(cos_table), _ptr(sin_table), _ptr(pos), _ptr(out),
                                                 _ptr(k_cache), _ptr(v_cache), _dt(qkv), n_head, n_kv_head, D, max_seq,
                                                 _ptr(workspace) if workspace is not None else None,
                                                 workspace.numel() * 4 if workspace is not None else 0, _stream()))


def prompt_attention(qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor, k_cache: torch.Tensor,
                     v_cache: torch.Tensor, n_head: int, n_kv_head: int, tables: bool = False) -> torch.Tensor:
    """Several tokens at once: qkv [S, (n_head + 2 n_kv_head) * D], cos / sin [S, D] (the tokens' rows; tables: the whole tables
    [max_seq, D], read at the positions; a row whose position they do not have comes out as no number), positions int64 [S] on the device;
    appends to the caches [1, n_kv_head, max_seq, D] and returns the attention output [S, n_head * D]."""
    _half_cuda(qkv, cos, sin, k_cache, v_cache)
    D, max_seq, S = k_cache.shape[-1], k_cache.shape[-2], qkv.shape[0]
    _check(qkv.dim() == 2 and qkv.shape[1] == (n_head + 2 * n_kv_head) * D, "qkv size mismatch")
    rows = max_seq if tables else S
    _check(tuple(cos.shape) == (rows, D) and tuple(sin.shape) == (rows, D), "cos and sin must be [rows, head_dim]")
    _check(positions.get_device() == qkv.get_device() and positions.is_contiguous() and positions.dtype == torch.int64 and positions.numel() == S,
           "positions must be one int64 per row on the device")
    _check(k_cache.numel() == n_kv_head * max_seq * D and v_cache.shape == k_cache.shape, "cache shape mismatch")
    q = torch.empty(S, n_head * D, dtype=qkv.dtype, device=qkv.device)
    out = torch.empty_like(q)
    lib = _lib.linears
    call = lib.decdec_prompt_attention_at if tables else lib.decdec_prompt_attention
    _lib.check(call(_ptr(qkv), _ptr(cos), _ptr(sin), _ptr(positions), _ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(out), _dt(qkv), S, n_head,
                    n_kv_head, D, max_seq, _stream()))
    return out


def dense_gemv(weight: torch.Tensor, x: torch.Tensor, out: torch.Tensor) -> None:
    """out[n] = sum_k weight[n, k] * x[k] for an unquantised fp16 / bf16 weight [N, K] (overwrites out)."""
    _half_cuda(weight, x, out)
    _check(weight.dim() == 2 and x.numel() == weight.shape[1] and out.numel() == weight.shape[0],
           "weight [N, K], x with K and out with N elements")
    _lib.check(_lib.linears.decdec_dense_gemv(_ptr(weight), _ptr(x), _ptr(out), _dt(out), weight.shape[0],
                                             weight.shape[1], _stream()))


def silu_mul(gate_up: torch.Tensor, out: torch.Tensor) -> None:
    _half_cuda(gate_up, out)
    _check(gate_up.numel() == 2 * out.numel(), "gate_up must hold twice as many elements as out")
    _lib.check(_lib.linears.decdec_silu_mul(_ptr(gate_up), _ptr(out), _dt(out), out.numel(), _stream()))


def silu_mul_rows(gate_up: torch.Tensor) -> torch.Tensor:
    """Rows [gate | up] of a prompt: gate_up [rows, 2 n] -> silu(gate) * up [rows, n]."""
    _half_cuda(gate_up)
    _check(gate_up.dim() == 2 and gate_up.shape[1] % 2 == 0, "gate_up must be [rows, 2 n]")
    rows, n = gate_up.shape[0], gate_up.shape[1] // 2
    out = torch.empty(rows, n, dtype=gate_up.dtype, device=gate_up.device)
    _lib.check(_lib.linears.decdec_silu_mul_rows(_ptr(gate_up), _ptr(out), _dt(out), rows, n, _stream()))
    return out


def add_rmsnorm(x: torch.Tensor, y, weight: torch.Tensor, h_out, normed_out: torch.Tensor, eps: float) -> None:
    """Rows of x [..., dim]: h = x + y (written to h_out; y = h_out = None: h = x), normed_out = rmsnorm(h) * weight."""
    ts = [t for t in (x, y, weight, h_out, normed_out) if t is not None]
    _half_cuda(*ts)
    dim = x.shape[-1]
    _check(weight.numel() == dim and normed_out.shape == x.shape, "weight / normed_out shape mismatch")
    _check((y is None) == (h_out is None) and (y is None or (y.shape == x.shape and h_out.shape == x.shape)),
           "y and h_out go together and have the shape of x")
    _lib.check(_lib.linears.decdec_add_rmsnorm(_ptr(x), _ptr(y) if y is not None else None, _ptr(weight),
                                              _ptr(h_out) if h_out is not None else None, _ptr(normed_out), _dt(x),
                                              x.numel() // dim, dim, float(eps), _stream()))


@functools.lru_cache(maxsize=1024)
def prompt_scratch_bytes(rows: int, dim: int, qkv: int, ff: int) -> int:
    """What `prompt_front` and `prompt_back` need between their kernels."""
    return int(_lib.load().decdec_prompt_scratch_bytes(rows, dim, qkv, ff))


def _prompt_part(call, dtype, rows, x, y, norm, eps, h, out, scratch, layers):
    numbers = [_DT[dtype], rows, x.data_ptr(), 0 if y is None else y.data_ptr(), norm.data_ptr(), 0 if h is None else h.data_ptr(), out.data_ptr(),
               scratch.data_ptr(), scratch.numel()]
    for layer in layers:
        numbers += layer
    part = array.array("Q", numbers + [0] * (33 - len(numbers)))           # decdec_prompt_part
    _lib.check(call(part.buffer_info()[0], float(eps), _stream()))


def prompt_front(x, y, norm, eps: float, layer, h, out, scratch) -> None:
    """Rows ahead of a block's attention: h = x + y (y = h = None: x), out = rmsnorm(h) times `layer` (linear.packed_layer).  scratch: bytes on the GPU."""
    _prompt_part(_lib.linears.decdec_prompt_front, x.dtype, out.shape[-2], x, y, norm, eps, h, out, scratch, (layer,))


def prompt_back(x, y, norm, eps: float, layers, h, out, scratch) -> None:
    """Rows behind a block's attention y: h = x + y Wo^T, out = the feed-forward of rmsnorm(h).  layers: Wo, gate and up, down (linear.packed_layer)."""
    _prompt_part(_lib.linears.decdec_prompt_back, x.dtype, out.shape[-2], x, y, norm, eps, h, out, scratch, layers)



def greedy_pick_workspace(device="cuda") -> torch.Tensor:
    """Workspace of `greedy_pick` (contents irrelevant; one serves any number of calls that do not overlap)."""
    return torch.empty(int(_lib.load().decdec_greedy_pick_workspace_bytes()) // 8, dtype=torch.int64, device=device)


def open_step(token, table, norm_weight, eps: float, h, normed, clear=None) -> None:
    """h = table[token], normed = rmsnorm(h) * norm_weight, and zeros in `clear`; token: one int64 on the device."""
    _half_cuda(table, norm_weight, h, normed)
    _pos(token, table)
    vocab, dim = table.shape
    _check(norm_weight.numel() == dim == h.numel() == normed.numel(), "norm_weight, h and normed must have as many elements as a row of the table")
    size = 0 if clear is None else clear.numel() * clear.element_size()
    _check(clear is None or (clear.get_device() == table.get_device() and clear.is_contiguous()), "clear must be a contiguous tensor of the same GPU")
    _lib.check(_lib.linears.decdec_open_step(_ptr(token), _ptr(table), _ptr(norm_weight), _ptr(h), _ptr(normed), None if clear is None else _ptr(clear), size,
                                            _dt(h), vocab, dim, float(eps), _stream()))


def product_makes(norm: bool, bits: int, dtype, K: int, N: int) -> bool:
    """Whether a SqueezeLLM product of one token may make its own activations (`norm_product`, `gate_product`).  Asked anew each time: the answer
    changes with the options that deal a product to workgroups."""
    return bool(_lib.linears.decdec_sqllm_step_fuses(norm, bits, _DT[dtype], K, N))


product_makes.__wrapped__ = product_makes                  # there is no cache to ask past


def norm_product(layer, x, y, norm, eps: float, h) -> torch.Tensor:
    """h = x + y (None both: x), the layer's output += its product of rmsnorm(h) * norm, in one launch.  `layer`: linear.step_layer holds."""
    _half_cuda(x, norm, layer.lut, layer.output, *((y, h) if y is not None else ()))
    K, N = layer.in_features, layer.out_features
    _check(x.numel() == norm.numel() == K and (y is None or y.numel() == h.numel() == K) and layer.output.numel() == N, "one row of the layer's input features")
    _lib.check(_lib.linears.decdec_sqllm_norm_gemv(_ptr(x), None if y is None else _ptr(y), _ptr(norm), float(eps), None if y is None else _ptr(h), _ptr(layer.output),
                                                  _ptr(layer.qweight), _ptr(layer.lut), layer.bitwidth, _dt(x), K, N, _stream()))
    return layer.output


def gate_product(layer, gate_up) -> torch.Tensor:
    """The layer's output += its product of silu(gate) * up, in one launch; gate_up: 2 in_features elements.  `layer`: linear.step_layer holds."""
    _half_cuda(gate_up, layer.lut, layer.output)
    K, N = layer.in_features, layer.out_features
    _check(gate_up.numel() == 2 * K and layer.output.numel() == N, "gate_up must be [2 in_features]")
    _lib.check(_lib.linears.decdec_sqllm_gate_gemv(_ptr(gate_up), _ptr(layer.output), _ptr(layer.qweight), _ptr(layer.lut), layer.bitwidth, _dt(gate_up), K, N, _stream()))
    return layer.output


def set_step(token: torch.Tensor, pos: torch.Tensor, count: torch.Tensor, first: int, at: int) -> None:
    """token = first, pos = at, count = 0: one int64 each, on the device."""
    for t in (token, pos, count):
        _check(t.get_device() == token.get_device() >= 0 and t.dtype is torch.int64 and t.numel() == 1, "token, pos and count must be one int64 each on one GPU")
    torch._C._increment_version((token, pos, count))     # an embedding that is still to be differentiated has kept the token
    _lib.check(_lib.linears.decdec_set_step(_ptr(token), _ptr(pos), _ptr(count), first, at, _stream()))


def greedy_pick(logits: torch.Tensor, workspace: torch.Tensor, token: torch.Tensor, seq=None, count=None, pos=None,
                logits_f32_out=None) -> None:
    """token[0] = argmax(logits) (smallest index among equal logits); seq[count[0]] = it and count[0] += 1 when seq and
    count are given; pos[0] += 1 when pos is given; logits_f32_out receives the logits as fp32 when given.  token, seq,
    count and pos are int64 tensors on the device."""
    _check(logits.is_cuda and logits.is_contiguous() and logits.dtype in (torch.float16, torch.bfloat16, torch.float32),
           "logits must be a contiguous fp16 / bf16 / fp32 CUDA tensor")
    for t in (token, seq, count, pos):
        _check(t is None or (t.is_cuda and t.is_contiguous() and t.dtype == torch.int64 and t.numel() >= 1),
               "token, seq, count and pos must be int64 CUDA tensors")
    _check((seq is None) == (count is None), "seq and count go together")
    _check(workspace.is_cuda and workspace.numel() * workspace.element_size() >= int(_lib.load().decdec_greedy_pick_workspace_bytes()),
           "workspace too small")
    _check(logits_f32_out is None or (logits_f32_out.is_cuda and logits_f32_out.is_contiguous() and
                                      logits_f32_out.dtype == torch.float32 and logits_f32_out.numel() >= logits.numel()),
           "logits_f32_out must be a contiguous fp32 CUDA tensor of at least as many elements")
    opt = lambda t: _ptr(t) if t is not None else None
    _lib.check(_lib.linears.decdec_greedy_pick(_ptr(logits), logits.numel(), _dt(logits), _ptr(workspace), opt(logits_f32_out),
                                              _ptr(token), opt(seq), seq.numel() if seq is not None else 0, opt(count),
                                              opt(pos), _stream()))
