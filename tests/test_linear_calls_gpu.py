"""A quantised layer called by itself: one call of the library clears the output where it has to, and multiplies."""
import ctypes

import pytest
import torch

from decdec_amd import ext
from decdec_amd.linear import APLinear, LUTGEMMLinear, SQLLMLinear
from test_prompt_linears_gpu import _layer

pytestmark = pytest.mark.gpu


def _call(fmt, config, x, out, packed):
    {"anyprec": ext.anyprec_linear, "lutgemm": ext.lutgemm_linear, "sqllm": ext.sqllm_linear}[fmt](config, x, out, *packed)


# one range of channels by the rule (called and captured, called only, by the outputs), several; outputs that are no multiple of two, of 64
SHAPES = [(32, 1), (512, 63), (1024, 1024), (1536, 65), (2048, 130), (3584, 200), (4096, 257), (5120, 64), (6144, 511), (8192, 12225), (14336, 96), (40960, 66)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("fmt,bits", [("sqllm", 3), ("sqllm", 4), ("lutgemm", 3), ("lutgemm", 4), ("lutgemm", 8), ("anyprec", 3), ("anyprec", 4), ("anyprec", 6)])
@pytest.mark.parametrize("K,N", SHAPES)
def test_output_is_overwritten(K, N, fmt, bits, dtype):
    if fmt == "anyprec" and dtype == torch.float32:
        pytest.skip("any-precision has no float32")
    torch.manual_seed(K + N)
    packed, dense = _layer(fmt, K, N, bits, 32, dtype)
    x = torch.randn(1, 1, K, device="cuda").to(dtype)
    want, size = (dense @ x.view(K).double()), dense.abs() @ x.view(K).double().abs()
    # a rounding of a range's sum for each of at most nine, of at most the sum of the terms' sizes; sums in float32
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -23}[dtype]
    bound = 10 * unit * (want.abs() + 3 * (dense.square() @ x.view(K).double().square()).sqrt()) + 2.0 ** -18 * size
    out = torch.full((1, 1, N), float("nan"), device="cuda", dtype=dtype)
    _call(fmt, None, x, out, packed)
    assert ((out.view(N).double() - want).abs() <= bound).all()
    again = torch.full_like(out, 7.0)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        _call(fmt, None, x, again, packed)
    for _ in range(3):
        again.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert ((again.view(N).double() - want).abs() <= bound).all()


def test_wrong_calls_are_refused():
    packed, _ = _layer("sqllm", 256, 64, 4, 32, torch.float16)
    x, out = torch.randn(1, 1, 256, device="cuda").half(), torch.zeros(1, 1, 64, device="cuda").half()
    for bad in [(x[:, :, :128], out, packed), (x.float(), out, packed), (x, out[:, :, :32], packed), (x.cpu(), out, packed), (x, out, (packed[0], packed[1], 5)),
                (x, out, (packed[0].long(), packed[1], 4)), (x.expand(1, 2, 256), out, packed), (x, out, (packed[0], packed[1].t().contiguous().t(), 4))]:
        with pytest.raises(RuntimeError):
            ext.sqllm_linear(None, bad[0], bad[1], *bad[2])
    with pytest.raises(RuntimeError, match="invalid DECConfig"):
        ext.sqllm_linear(12345, x, out, *packed)


def test_sizes_that_a_file_has_as_floats():
    (q, alpha, bias, bits, group), _ = _layer("lutgemm", 512, 96, 3, 64, torch.float16)
    x, a, b = torch.randn(1, 1, 512, device="cuda").half(), torch.zeros(1, 1, 96, device="cuda").half(), torch.zeros(1, 1, 96, device="cuda").half()
    ext.lutgemm_linear(None, x, a, q, alpha, bias, bits, group)
    ext.lutgemm_linear(None, x, b, q, alpha, bias, float(bits), float(group))
    assert torch.equal(a, b)


def test_numbers_of_heads_that_are_floats_are_refused():
    from decdec_amd import decode_ops
    H, KV, D, S = 4, 2, 64, 16
    make = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.float16)
    qkv, cos, sin, out, k, v = make((H + 2 * KV) * D), make(S, D), make(S, D), make(H * D), make(KV, S, D), make(KV, S, D)
    pos = torch.zeros(1, dtype=torch.int64, device="cuda")
    decode_ops.rope_attention(qkv, cos, sin, pos, out, k, v, H, KV)
    for heads in ((float(H), KV), (H, float(KV))):
        with pytest.raises(ctypes.ArgumentError):
            decode_ops.rope_attention(qkv, cos, sin, pos, out, k, v, *heads)


def _module(fmt, K, N):
    packed, _ = _layer(fmt, K, N, 3, 32, torch.float16)
    if fmt == "anyprec":
        layer = APLinear(K, N, 3)
        layer.qweight, layer.lut = packed[:2]
    elif fmt == "lutgemm":
        layer = LUTGEMMLinear(K, N, 3, 32)
        layer.qweight, layer.alpha, layer.q_bias = packed[:3]
    else:
        layer = SQLLMLinear(K, N, 3)
        layer.qweight, layer.lut = packed[:2]
    return layer


@pytest.mark.parametrize("fmt", ["anyprec", "lutgemm", "sqllm"])
def test_a_result_that_is_overwritten_is_not_differentiated(fmt):
    """A layer keeps one output: what autograd has saved of it is gone with the next call, in whatever mode that is made."""
    layer, p = _module(fmt, 1024, 96), torch.ones(96, device="cuda", dtype=torch.float16, requires_grad=True)
    x = torch.randn(2, 1, 1, 1024, device="cuda", dtype=torch.float16)
    y = layer(x[0]).clone()
    (layer(x[0]) * p).sum().backward()
    # sums of ranges may be added in another order
    assert ((p.grad - y.view(-1)).abs() <= 0.02 * y.abs().max()).all()
    for mode in (torch.enable_grad, torch.no_grad, torch.inference_mode):
        loss = (layer(x[0]) * p).sum()
        with mode():
            layer(x[1])
        with pytest.raises(RuntimeError, match="inplace operation"):
            loss.backward()


@pytest.mark.parametrize("fmt", ["anyprec", "lutgemm", "sqllm"])
def test_a_bias_that_is_learnt_has_the_gradient_of_the_last_call(fmt):
    layer, x = _module(fmt, 512, 64), torch.randn(1, 1, 512, device="cuda", dtype=torch.float16)
    layer.bias = torch.nn.Parameter(torch.zeros(64, device="cuda", dtype=torch.float16))
    for _ in range(3):
        layer.bias.grad = None
        layer(x).sum().backward()
        assert torch.equal(layer.bias.grad, torch.ones_like(layer.bias))
