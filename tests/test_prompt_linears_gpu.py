"""Quantised linears over several tokens: dense weights out of the packed formats."""
import pytest
import torch

from decdec_amd import ext, formats as F

pytestmark = pytest.mark.gpu


def _words(*shape):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int64).to(torch.int32).cuda()


# edges: tiles of 64 outputs x 128 channels, units of 32 channels, one output, more tiles than workgroups along K
SHAPES = [(32, 1), (96, 63), (128, 64), (160, 65), (2080, 130), (33 * 128, 200)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bits", [3, 4])
@pytest.mark.parametrize("K,N", SHAPES)
def test_sqllm_dequant_is_the_table_lookup(K, N, bits, dtype):
    torch.manual_seed(K + N)
    q, lut = _words(K * bits // 32, N), torch.randn(N, 2 ** bits, device="cuda").to(dtype)
    assert torch.equal(ext.sqllm_dequant(q, lut, bits), F.dequant_sqllm(q, lut, bits))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bits,group", [(1, 32), (2, 16), (3, 128), (4, 32), (5, 8), (8, 64)])
@pytest.mark.parametrize("K,N", [(128, 1), (256, 65), (1152, 130)])
def test_lutgemm_dequant_is_the_signed_sum(K, N, bits, group, dtype):
    torch.manual_seed(K + N)
    q, alpha = _words(K // 32, bits, N), torch.rand(K // group, bits, N, device="cuda").to(dtype)
    bias = torch.randn(K // group, N, device="cuda").to(dtype)
    got = ext.lutgemm_dequant(q, alpha, bias, bits, group).double()
    want = F.dequant_bcq(q, alpha, bias, group).double()
    # fp32 sums of bits + 1 terms of size at most `big` in another order, then one rounding to the storage type
    big = alpha.double().sum(1).max() + bias.double().abs().max()
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[dtype]
    assert ((got - want).abs() <= unit * want.abs() + (bits + 1) * 2.0 ** -23 * big).all()


def test_dequant_refuses_what_does_not_fit():
    q, lut = _words(8, 16), torch.zeros(16, 16, device="cuda", dtype=torch.float16)
    with pytest.raises(RuntimeError):
        ext.sqllm_dequant(q, lut, 5)
    with pytest.raises(RuntimeError):
        ext.sqllm_dequant(q, lut[:8], 4)
    with pytest.raises(RuntimeError):
        ext.lutgemm_dequant(_words(4, 3, 16), torch.zeros(2, 3, 16, device="cuda"), torch.zeros(2, 16, device="cuda"), 3, 48)
