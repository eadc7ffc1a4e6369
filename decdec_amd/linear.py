"""nn.Module front ends of the ops, with the interface of the reference's end-to-end modules.

``DECLinear`` / ``APLinear`` / ``LUTGEMMLinear`` follow the reference's end-to-end/DECLinear.py,
APLinear.py and LUTGEMMLinear.py (same constructor arguments, buffers, ``load_dec_data`` /
``create_dec_config`` / ``update_dec_config`` methods, decode path = the product in the persistent output
buffer (cleared inside the call where workgroups add to it), prefill path = dequantise + matmul).  ``SQLLMLinear`` is the same
pattern for the ``dec_sqllm`` op, for which the reference ships no module.
"""
from __future__ import annotations

import torch
import torch.nn as nn

from . import decode_ops, ext, formats


# Prompts of at most PACKED_TOKENS tokens multiply with the packed weight, longer ones with its dense expansion: decoding is repeated
# for every 128 tokens, expanding is not.  SqueezeLLM and 3-bit LUT-GEMM, which decode fastest, multiply large layers packed up to twice
# as many.  Packed / dense, us, fp16, graphs of layers one after another, at 256, 300, 384, 448 and 512 tokens:
#   SqueezeLLM 4 bits     4096 -> 28672 83/147 84/151 89/155 101/172 109/164, 4096 -> 4096 27/32 29/35 31/35 31/39 32/39
#   SqueezeLLM 3 bits     4096 -> 28672 73/143 72/148 82/146 94/165 107/168, 14336 -> 4096 46/92 65/99 69/104 67/116 73/118
#   LUT-GEMM 3 bits       4096 -> 28672 80/145 75/151 85/150 97/165 152/167, 14336 -> 4096 48/95 68/102 74/103 69/118 75/120
#   LUT-GEMM 4 bits       4096 -> 28672 104/142 137/145 149/155 180/168 189/166, 4096 -> 6144 35/50 44/40 48/45 47/46 51/47
#   any-precision 3 bits  4096 -> 28672 87/138 110/143 121/151 153/165 163/163, 4096 -> 4096 28/29 31/33 33/33 34/37 36/37
#   any-precision 4 bits  4096 -> 28672 103/139 133/145 142/155 175/169 192/166, 4096 -> 6144 38/50 46/40 49/44 49/45 52/47
# (the first three at 4096 -> 28672 from 300 tokens on in wide tiles, k_qgemm_wide.hip).  The line of the other three was drawn when they were even at 300 tokens; the largest
# layers would gain up to 384 or 448 by now, those of 4096 -> 6144 lose from 300 on.  Layers of fewer weights are bound by their launches either way.
PACKED_TOKENS, LARGE = 256, 1 << 24


def _packed_tokens(fmt: str, bitwidth: int, weights: int) -> int:
    twice = weights >= LARGE and (fmt == "sqllm" or (fmt == "lutgemm" and bitwidth == 3))
    return 2 * PACKED_TOKENS if twice else PACKED_TOKENS


def _packed(x, bitwidth, most, *tensors) -> bool:
    """Whether a prompt's product runs on the packed weight, with at most `most` tokens (autocast chooses a torch product's type, which
    may not be x's)."""
    if (x.dim() != 3 or x.shape[0] != 1 or x.shape[1] > most or bitwidth not in (3, 4) or x.dtype not in (torch.float16, torch.bfloat16)
            or x.dtype != tensors[1].dtype or torch.is_autocast_enabled()):
        return False
    at, table = x.data_ptr(), tensors[1].data_ptr()        # 0: no tokens, channels or outputs
    return at > 0 and table > 0 and (at | table) % 16 == 0 and ext.on_kernels(x.device, x, *tensors)


def packed_layer(l, rows: int, dtype, index: int):
    """A layer as the library takes it in a part of a prompt (decdec_packed_layer, in its order), or None: `l` is of another class than those here, somebody
    sees or changes its calls, or `rows` tokens of `dtype` on GPU `index` are not multiplied packed.  Nothing watches torch operations, and the GPU is the
    current one."""
    kind = _KINDS.get(type(l))
    if kind is None or l._forward_hooks or l._forward_pre_hooks or "forward" in l.__dict__ or "gemm" in l.__dict__ or l.bias is not None:
        return None
    buffers, bits, K, N = l._buffers, l.bitwidth, l.in_features, l.out_features
    q, group, last = buffers.get("qweight"), 0, 0
    if kind == 1:
        table, group, bias = buffers.get("alpha"), l.group_size, buffers.get("q_bias")
        if table is None or bias is None or group % 32 or K % group or table.shape != (K // group, bits, N) or bias.shape != (K // group, N) or bias.dtype != dtype \
                or not ext.plain(index, bias):
            return None
        last = bias.data_ptr()
    else:
        table = buffers.get("lut")
        if table is None or table.shape != (N, 1 << bits):
            return None
    if (bits != 3 and bits != 4) or K % 32 or q is None or table.dtype != dtype or q.dtype != torch.int32 or rows > _packed_tokens(_FORMATS[kind], bits, K * N) \
            or q.shape != ((bits, N, K // 32), (K // 32, bits, N), (K * bits // 32, N))[kind] or not ext.plain(index, q, table):
        return None
    at = table.data_ptr()
    return None if at == 0 or at % 16 else (kind, bits, group, K, N, q.data_ptr(), at, last)


def may_make(l) -> bool:
    """Whether a layer is of those that `step_layer` asks more of: of this class, uncompensated, with an output that is cleared elsewhere."""
    return type(l) is SQLLMLinear and l.dec_config is None and l.external_zero


def step_layer(l, norm: bool, dtype, index: int) -> bool:
    """Whether a layer's product of one token may make its own activations (`decode_ops.norm_product`, `gate_product`): of this class, nobody sees its calls, no
    compensation (which selects among the activations), an output that is cleared elsewhere, plain tensors on GPU `index`."""
    if not may_make(l) or l._forward_hooks or l._forward_pre_hooks or "forward" in l.__dict__ or l.bias is not None or l.bitwidth not in (3, 4):
        return False
    q, lut, out, K, N = l._buffers.get("qweight"), l._buffers.get("lut"), l.output, l.in_features, l.out_features
    return (q is not None and lut is not None and lut.dtype == out.dtype == dtype and q.dtype == torch.int32 and K % 32 == 0 and ext.plain(index, q, lut, out)
            and q.shape == (K * l.bitwidth // 32, N) and lut.shape == (N, 1 << l.bitwidth) and out.shape == (1, 1, N) and lut.data_ptr() % 16 == 0
            and out.data_ptr() % 4 == 0 and decode_ops.product_makes(norm, l.bitwidth, dtype, K, N))


class DECLinear(nn.Module):
    """Holds the DEC side data of a quantised linear layer (reference DECLinear.py:6-53)."""

    def __init__(self):
        super().__init__()
        self.dec_config = None
        self.k_chunk = None
        self.q_residual = None
        self.scales = None
        self.thresholds = None
        self.external_zero = False      # True: the owner of `output` clears it before every decode step

    def load_dec_data(self, q_residual, scales, thresholds):
        assert q_residual.dtype == torch.int
        assert q_residual.shape == (self.in_features, self.out_features // 8)
        assert scales.dtype == self.dtype
        assert scales.shape == (self.out_features,)
        assert thresholds.dtype == self.dtype
        assert thresholds.shape == (self.in_features,)
        self.q_residual = q_residual
        self.scales = scales
        self.thresholds = thresholds

    def create_dec_config(self, dec_context, k_chunk):
        self.k_chunk = k_chunk
        assert self.q_residual is not None and self.scales is not None and self.thresholds is not None
        self.dec_config = ext.create_dec_config(dec_context, k_chunk, self.q_residual, self.scales, self.thresholds)

    def update_dec_config(self, dec_context, k_chunk):
        """New context / k_chunk without copying the residual again."""
        self.k_chunk = k_chunk
        assert self.dec_config is not None
        ext.update_dec_config(self.dec_config, dec_context, k_chunk)

    def _finish(self):
        if self.bias is not None:
            self.output += self.bias
        return self.output


class APLinear(DECLinear):
    """Any-precision bitplane layer (reference APLinear.py:7-58)."""

    def __init__(self, in_features, out_features, bitwidth, bias=False, dtype=torch.half, device="cuda"):
        super().__init__()
        self.in_features, self.out_features, self.bitwidth, self.dtype = in_features, out_features, bitwidth, dtype
        self.register_buffer("qweight", torch.empty((bitwidth, out_features, in_features // 32),
                                                    dtype=torch.int32, device=device))
        self.register_buffer("lut", torch.empty((out_features, 2 ** bitwidth), dtype=dtype, device=device))
        if bias:
            self.register_buffer("bias", torch.empty((out_features,), dtype=dtype, device=device))
        else:
            self.bias = None
        self.output = torch.zeros((1, 1, out_features), dtype=dtype, device=device)

    def gemm(self, x):
        if _packed(x, self.bitwidth, PACKED_TOKENS, self.qweight, self.lut):
            return ext.anyprec_gemm(x[0], self.qweight, self.lut, self.bitwidth)[None]
        weight = ext.anyprec_dequant(self.qweight, self.lut, self.bitwidth)
        return torch.matmul(x, weight.T)

    def forward(self, x, **kwargs):
        assert x.shape[0] == 1
        if x.shape[1] > 1:
            out = self.gemm(x)
            if self.bias is not None:
                out += self.bias
            return out
        if not self.external_zero:
            ext.anyprec_linear(self.dec_config, x, self.output, self.qweight, self.lut, self.bitwidth)
        elif self.dec_config is None:
            ext.anyprec_gemv(x, self.output, self.qweight, self.lut, self.bitwidth)
        else:
            ext.dec_anyprec(self.dec_config, x, self.output, self.qweight, self.lut, self.bitwidth)
        return self._finish()


class LUTGEMMLinear(DECLinear):
    """LUT-GEMM binary-coding layer (reference LUTGEMMLinear.py:6-102)."""

    def __init__(self, in_features, out_features, bitwidth, group_size, bias=False, dtype=torch.half, device="cuda"):
        super().__init__()
        self.in_features, self.out_features = in_features, out_features
        self.bitwidth, self.group_size, self.dtype = bitwidth, group_size, dtype
        self.register_buffer("qweight", torch.empty((in_features // 32, bitwidth, out_features),
                                                    dtype=torch.int32, device=device))
        self.register_buffer("alpha", torch.empty((in_features // group_size, bitwidth, out_features),
                                                  dtype=dtype, device=device))
        self.register_buffer("q_bias", torch.empty((in_features // group_size, out_features),
                                                   dtype=dtype, device=device))
        if bias:
            self.register_buffer("bias", torch.empty((out_features,), dtype=dtype, device=device))
        else:
            self.bias = None
        self.output = torch.zeros((1, 1, out_features), dtype=dtype, device=device)

    def gemm(self, x):
        if self.group_size % 32 == 0 and self.in_features % self.group_size == 0 \
                and _packed(x, self.bitwidth, _packed_tokens("lutgemm", self.bitwidth, self.in_features * self.out_features),
                            self.qweight, self.alpha, self.q_bias):
            return ext.lutgemm_gemm(x[0], self.qweight, self.alpha, self.q_bias, self.bitwidth, self.group_size)[None]
        if x.dtype == self.alpha.dtype == self.q_bias.dtype and x.dtype in ext._DT and self.qweight.numel() and self.in_features % self.group_size == 0 \
                and ext.on_kernels(x.device, self.qweight, self.alpha, self.q_bias):
            weight = ext.lutgemm_dequant(self.qweight, self.alpha, self.q_bias, self.bitwidth, self.group_size)
        else:
            weight = formats.dequant_bcq(self.qweight, self.alpha, self.q_bias, self.group_size).to(x.dtype)
        return torch.matmul(x, weight.T)

    def forward(self, x, **kwargs):
        assert x.shape[0] == 1
        if x.shape[1] > 1:
            out = self.gemm(x)
            if self.bias is not None:
                out += self.bias
            return out
        if not self.external_zero:
            ext.lutgemm_linear(self.dec_config, x, self.output, self.qweight, self.alpha, self.q_bias, self.bitwidth, self.group_size)
        elif self.dec_config is None:
            ext.lutgemm_gemv(x, self.output, self.qweight, self.alpha, self.q_bias, self.bitwidth, self.group_size)
        else:
            ext.dec_lutgemm(self.dec_config, x, self.output, self.qweight, self.alpha, self.q_bias,
                            self.bitwidth, self.group_size)
        return self._finish()


class SQLLMLinear(DECLinear):
    """SqueezeLLM per-channel LUT layer over the ``sqllm_gemv`` / ``dec_sqllm`` ops."""

    def __init__(self, in_features, out_features, bitwidth, bias=False, dtype=torch.half, device="cuda"):
        super().__init__()
        self.in_features, self.out_features, self.bitwidth, self.dtype = in_features, out_features, bitwidth, dtype
        self.register_buffer("qweight", torch.empty((in_features * bitwidth // 32, out_features),
                                                    dtype=torch.int32, device=device))
        self.register_buffer("lut", torch.empty((out_features, 2 ** bitwidth), dtype=dtype, device=device))
        if bias:
            self.register_buffer("bias", torch.empty((out_features,), dtype=dtype, device=device))
        else:
            self.bias = None
        self.output = torch.zeros((1, 1, out_features), dtype=dtype, device=device)

    def gemm(self, x):
        # the kernels decode 32 channels at a time; 4 bits may hold fewer
        units = self.in_features % 32 == 0 and self.qweight.numel() > 0
        if units and _packed(x, self.bitwidth, _packed_tokens("sqllm", self.bitwidth, self.in_features * self.out_features), self.qweight, self.lut):
            return ext.sqllm_gemm(x[0], self.qweight, self.lut, self.bitwidth)[None]
        if units and self.lut.dtype in ext._DT and ext.on_kernels(x.device, self.qweight, self.lut):
            weight = ext.sqllm_dequant(self.qweight, self.lut, self.bitwidth)
        else:
            weight = formats.dequant_sqllm(self.qweight, self.lut, self.bitwidth)
        return torch.matmul(x, weight.T)

    def forward(self, x, **kwargs):
        assert x.shape[0] == 1
        if x.shape[1] > 1:
            out = self.gemm(x)
            if self.bias is not None:
                out += self.bias
            return out
        if not self.external_zero:
            ext.sqllm_linear(self.dec_config, x, self.output, self.qweight, self.lut, self.bitwidth)
        elif self.dec_config is None:
            ext.sqllm_gemv(x, self.output, self.qweight, self.lut, self.bitwidth)
        else:
            ext.dec_sqllm(self.dec_config, x, self.output, self.qweight, self.lut, self.bitwidth)
        return self._finish()


_KINDS, _FORMATS = {APLinear: 0, LUTGEMMLinear: 1, SQLLMLinear: 2}, ("anyprec", "lutgemm", "sqllm")
