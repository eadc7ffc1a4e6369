"""Quantised linears over several tokens: dense weights out of the packed formats."""
import ctypes

import pytest
import torch

from decdec_amd import _lib, ext, formats as F

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
@pytest.mark.parametrize("bits,group", [(1, 32), (2, 16), (3, 128), (3, 8), (4, 32), (4, 64), (5, 8), (8, 64)])
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


def _layer(fmt, K, N, bits, group, dtype):
    """(packed tensors, dense weight in fp64) of a random layer."""
    if fmt == "lutgemm":
        q, alpha = _words(K // 32, bits, N), (torch.rand(K // group, bits, N, device="cuda") * 0.1).to(dtype)
        bias = (torch.randn(K // group, N, device="cuda") * 0.1).to(dtype)
        return (q, alpha, bias, bits, group), F.dequant_bcq(q, alpha, bias, group).to(dtype).double()
    lut = torch.randn(N, 2 ** bits, device="cuda").to(dtype)
    if fmt == "sqllm":
        q = _words(K * bits // 32, N)
        return (q, lut, bits), F.dequant_sqllm(q, lut, bits).double()
    q = _words(bits, N, K // 32)
    return (q, lut, bits), F.dequant_lut(F.unpack_anyprec(q, bits), lut).double()


# tokens at the edges of every instance (multiples of 16 up to 128) and of two and three token tiles; channels of less than a packet of
# 128, of a block of 512 and of an any-precision chunk of 1024, and with ranges in several workgroups; odd and single outputs
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt,bits", [("anyprec", 3), ("anyprec", 4), ("lutgemm", 3), ("lutgemm", 4), ("sqllm", 3), ("sqllm", 4)])
@pytest.mark.parametrize("M,K,N", [(2, 32, 1), (2, 4096, 1024), (16, 1120, 65), (17, 512, 130), (33, 2080, 64), (48, 3072, 96), (49, 96, 257),
                                   (64, 1024, 130), (65, 2080, 72), (80, 5120, 200), (81, 1056, 128), (96, 544, 264), (97, 2048, 33),
                                   (112, 4096, 66), (113, 96, 520), (128, 2048, 72), (129, 640, 40), (300, 1024, 136)])
def test_product_with_a_packed_weight(M, K, N, fmt, bits, dtype):
    torch.manual_seed(M + K + N)
    group = 32 if K % 64 else 64
    args, w = _layer(fmt, K, N, bits, group, dtype)
    x = torch.randn(M, K, device="cuda").to(dtype)
    got = getattr(ext, f"{fmt}_gemm")(x, *args).double()
    want = x.double() @ w.T.contiguous()
    # fp32 sums of K terms (their error grows like the square root of K here) and one rounding; a LUT-GEMM value whose fp32 sum
    # is taken in another order may round the other way (one unit of a weight, K times)
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    size = (x.double().square() @ w.T.square().contiguous()).sqrt()
    assert ((got - want).abs() <= unit * want.abs() + (2.0 ** -19 + (unit / 2 if fmt == "lutgemm" else 0)) * size + 1e-30).all()


def _form(fmt, bits, group, M, K, N):
    out = ctypes.c_int(-1)
    _lib.check(_lib.load().decdec_quant_gemm_form({"anyprec": 0, "lutgemm": 1, "sqllm": 2}[fmt], bits, group, M, K, N, ctypes.byref(out)))
    return out.value


# Tiles of 256 tokens x 256 outputs: tokens at the edges of every instance, one and two token tiles, one block of channels and several (odd and
# even), the fewest and the most outputs that fill a turn, outputs that are no multiple of 8, of 32 and of 256, the turn after; four and eight
# token tiles whose last one is ragged, groups of 256 and 384 channels; one token and one output less than goes there, one block of channels
# in two turns and in a turn that is not full
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt,bits", [("sqllm", 4), ("sqllm", 3), ("lutgemm", 3)])
@pytest.mark.parametrize("M,K,N,group,wide", [
    (257, 512, 22529, 128, True), (288, 1024, 22600, 256, True), (320, 512, 32768, 128, True), (321, 1536, 24580, 384, True), (384, 512, 24576, 128, True),
    (385, 1024, 23013, 128, True), (448, 1024, 22664, 128, True), (449, 512, 28672, 128, True), (512, 1536, 28672, 128, True), (512, 1024, 22528, 128, False),
    (256, 512, 28672, 128, False), (160, 512, 49153, 128, True), (145, 512, 49160, 128, True), (300, 1024, 49153, 128, True), (777, 1024, 28672, 256, True),
    (770, 1536, 12313, 384, True), (1999, 1024, 6144, 128, True), (1793, 512, 6150, 128, True), (129, 512, 49160, 128, True), (128, 512, 49160, 128, False),
    (777, 512, 24576, 128, False), (257, 512, 49153, 128, False), (448, 512, 24576, 128, False), (448, 512, 26625, 128, True)])
def test_product_in_wide_tiles(M, K, N, group, wide, fmt, bits, dtype):
    torch.manual_seed(M + K + N)
    # LUT-GEMM's sums and a decoded packet of 16 tiles of tokens do not fit the registers
    tiles = -(-M // -(-M // 256))
    assert _form(fmt, bits, group, M, K, N) == int(wide and (fmt == "sqllm" or tiles <= 224))
    args, w = _layer(fmt, K, N, bits, group, dtype)
    x = torch.randn(M, K, device="cuda").to(dtype)
    got = getattr(ext, f"{fmt}_gemm")(x, *args).double()
    want = x.double() @ w.T.contiguous()
    # the bound of the test above
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    size = (x.double().square() @ w.T.square().contiguous()).sqrt()
    assert ((got - want).abs() <= unit * want.abs() + (2.0 ** -19 + (unit / 2 if fmt == "lutgemm" else 0)) * size + 1e-30).all()


# LUT-GEMM groups that a lane's table serves for a whole block, with channels that end inside a block of 512; several turns of whole tiles;
# several token tiles whose columns are dealt to dies, with a number of column groups that eight does not divide, split and not; long rows
# split among workgroups
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt,bits,group", [("anyprec", 3, 0), ("lutgemm", 3, 128), ("lutgemm", 4, 256), ("sqllm", 4, 0)])
@pytest.mark.parametrize("M,K,N", [(16, 1280, 40), (3, 2048, 33000), (40, 1280, 33100), (77, 4352, 136), (160, 1280, 1100), (300, 2304, 1048),
                                   (512, 1536, 2056)])
def test_product_dealt_in_whole_and_split_tiles(M, K, N, fmt, bits, group, dtype):
    torch.manual_seed(M + K + N)
    args, w = _layer(fmt, K, N, bits, group, dtype)
    x = torch.randn(M, K, device="cuda").to(dtype)
    got = getattr(ext, f"{fmt}_gemm")(x, *args).double()
    want = x.double() @ w.T.contiguous()
    # the bound of the test above
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    size = (x.double().square() @ w.T.square().contiguous()).sqrt()
    assert ((got - want).abs() <= unit * want.abs() + (2.0 ** -19 + (unit / 2 if fmt == "lutgemm" else 0)) * size + 1e-30).all()


def _tiles(M, N):
    """(workgroup tiles of a product, bytes of a tile's sums in 32 bits)."""
    mt = -(-(-(-M // -(-M // 128))) // 16)
    columns, z = (128 if mt >= 3 else 64), -(-M // (16 * mt))
    groups = -(-N // columns)
    return (groups if z == 1 else -(-groups // 8) * 8 * z), 16 * mt * columns * 4


# Full turns of whole tiles (512 of 64 outputs for one tile of tokens, 256 of 128 outputs for three and more) and a split rest behind them, of
# one and of two token tiles: `split` tiles in `ks` shares each
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt,bits", [("anyprec", 3), ("lutgemm", 3), ("lutgemm", 4), ("sqllm", 4)])
@pytest.mark.parametrize("M,K,N,split,ks", [(3, 4096, 33000, 4, 2), (40, 2048, 33100, 3, 2), (130, 4096, 33000, 16, 4), (160, 2048, 16500, 16, 2)])
def test_product_of_whole_tiles_and_a_split_rest(M, K, N, split, ks, fmt, bits, dtype):
    from decdec_amd import _lib
    tiles, size = _tiles(M, N)
    assert tiles > split and int(_lib.load().decdec_quant_gemm_workspace_bytes(M, K, N)) == split * ks * size
    torch.manual_seed(M + N)
    args, w = _layer(fmt, K, N, bits, 128, dtype)
    x = torch.randn(M, K, device="cuda").to(dtype)
    got = getattr(ext, f"{fmt}_gemm")(x, *args).double()
    want = x.double() @ w.T.contiguous()
    # the bound of the tests above
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    spread = (x.double().square() @ w.T.square().contiguous()).sqrt()
    assert ((got - want).abs() <= unit * want.abs() + (2.0 ** -19 + (unit / 2 if fmt == "lutgemm" else 0)) * spread + 1e-30).all()


# Rows whose offsets within a tile of tokens need one tile (2^24 channels), and a row at a time (2^27), to have 32 bits
@pytest.mark.parametrize("M,K,N", [(20, 2 ** 24 + 64, 40), (2, 2 ** 27 + 64, 2)])
def test_product_of_very_long_rows(M, K, N):
    g = torch.Generator(device="cuda").manual_seed(M)
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), generator=g, device="cuda", dtype=torch.int32)
    lut = torch.randn(N, 16, generator=g, device="cuda").half()
    x = (torch.randn(M, K, generator=g, device="cuda", dtype=torch.float16) * 0.25)
    got, want, square = ext.sqllm_gemm(x, q, lut, 4).double(), 0.0, 0.0
    step = 2 ** 22
    for at in range(0, K, step):
        w, part = F.dequant_sqllm(q[at // 8:(at + step) // 8], lut, 4).double().T.contiguous(), x[:, at:at + step].double()
        want, square = want + part @ w, square + part.square() @ w.square()
    # fp32 sums of K / 32 products of 32 in at most 64 ranges (their error grows like the square root of a range's number, four times that), one rounding
    assert ((got - want).abs() <= 2.0 ** -11 * want.abs() + 4 * (K / 32) ** 0.5 * 2.0 ** -24 * square.sqrt() + 1e-30).all()


@pytest.mark.parametrize("fmt,bits", [("sqllm", 3), ("sqllm", 4), ("lutgemm", 3)])
def test_product_of_very_many_outputs(fmt, bits):
    """From 2^24 outputs on the offsets within a block of words do not have 32 bits."""
    M, K, N, step = 3, 64, 2 ** 24 + 8, 2 ** 20
    g = torch.Generator(device="cuda").manual_seed(bits)
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31 - 1, s, generator=g, device="cuda", dtype=torch.int32)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    if fmt == "sqllm":
        q, lut = words(K * bits // 32, N), torch.randn(N, 2 ** bits, generator=g, device="cuda").half()
        got, weight = ext.sqllm_gemm(x, q, lut, bits), lambda at: F.dequant_sqllm(q[:, at:at + step].contiguous(), lut[at:at + step], bits)
    else:
        q, alpha = words(K // 32, bits, N), (torch.rand(1, bits, N, generator=g, device="cuda") * 0.1).half()
        bias = (torch.randn(1, N, generator=g, device="cuda") * 0.1).half()
        part = lambda t, at: t[..., at:at + step].contiguous()
        got, weight = ext.lutgemm_gemm(x, q, alpha, bias, bits, K), lambda at: F.dequant_bcq(part(q, at), part(alpha, at), part(bias, at), K).half()
    for at in range(0, N, step):
        w = weight(at).double().T.contiguous()
        want, size = x.double() @ w, (x.double().square() @ w.square()).sqrt()
        # the bound of the tests above
        assert ((got[:, at:at + step].double() - want).abs() <= 2.0 ** -11 * want.abs() + (2.0 ** -19 + (2.0 ** -12 if fmt == "lutgemm" else 0)) * size + 1e-30).all()


@pytest.mark.parametrize("fmt,bits,most", [("sqllm", 4, 512), ("lutgemm", 3, 512), ("lutgemm", 4, 256), ("anyprec", 3, 256)])
def test_large_layers_multiply_packed_up_to(fmt, bits, most, monkeypatch):
    from decdec_amd import linear
    taken = []
    for name in (f"{fmt}_gemm", f"{fmt}_dequant"):
        monkeypatch.setattr(ext, name, lambda *a, name=name: taken.append(name) or torch.zeros(4096, 4096, device="cuda", dtype=torch.float16))
    layer = (linear.LUTGEMMLinear(4096, 4096, bits, 128) if fmt == "lutgemm" else (linear.APLinear if fmt == "anyprec" else linear.SQLLMLinear)(4096, 4096, bits))
    for tokens in (most, most + 1):
        layer(torch.zeros(1, tokens, 4096, device="cuda", dtype=torch.float16))
    assert taken == [f"{fmt}_gemm", f"{fmt}_dequant"]


@pytest.mark.parametrize("fmt", ["anyprec", "lutgemm", "sqllm"])
def test_product_takes_unaligned_packed_words(fmt):
    """Words and scales that start at an odd element are read one by one."""
    torch.manual_seed(0)
    args, w = _layer(fmt, 1024, 64, 3, 128, torch.float16)
    odd = torch.zeros(args[0].numel() + 1, dtype=torch.int32, device="cuda")[1:].view(args[0].shape)
    odd.copy_(args[0])
    x = torch.randn(20, 1024, device="cuda", dtype=torch.float16)
    assert torch.equal(getattr(ext, f"{fmt}_gemm")(x, odd, *args[1:]), getattr(ext, f"{fmt}_gemm")(x, *args))


def test_product_into_an_output_that_starts_anywhere():
    """Ranges of channels of different workgroups, summed into results that start at an odd element, through the C interface."""
    from decdec_amd import _lib
    torch.manual_seed(1)
    M, K, N = 16, 4096, 64
    (q, lut, bits), _ = _layer("sqllm", K, N, 4, 128, torch.float16)
    x, lib = torch.randn(M, K, device="cuda", dtype=torch.float16), _lib.load()
    need = int(lib.decdec_quant_gemm_workspace_bytes(M, K, N))
    assert need > 0
    room, ws = torch.full((M * N + 16,), 7.0, device="cuda", dtype=torch.float16), torch.empty(need, device="cuda", dtype=torch.uint8)
    for first in (1, 3, 4, 8):
        out = room.fill_(7.0)[first:first + M * N]
        _lib.check(lib.decdec_quant_gemm(2, x.data_ptr(), out.data_ptr(), q.data_ptr(), lut.data_ptr(), None, bits, 0, 1, M, K, N, ws.data_ptr(), need,
                                         torch.cuda.current_stream().cuda_stream))
        assert torch.equal(out.view(M, N), ext.sqllm_gemm(x, q, lut, bits))
        assert (room[:first] == 7.0).all() and (room[first + M * N:] == 7.0).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n", [(2, 8), (3, 13), (77, 17920), (5, 264)])
def test_silu_mul_of_rows(rows, n, dtype):
    from decdec_amd import decode_ops
    torch.manual_seed(n)
    gu = (torch.randn(rows, 2 * n, device="cuda") * 3).to(dtype)
    want = torch.nn.functional.silu(gu[:, :n].double()) * gu[:, n:].double()
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8            # one rounding, fp32 with a fast exponential before it
    assert ((decode_ops.silu_mul_rows(gu).double() - want).abs() <= (unit + 2.0 ** -20) * want.abs() + 2.0 ** -24).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [3, 4, 5])
@pytest.mark.parametrize("K,N", SHAPES)
def test_anyprec_dequant_is_the_table_lookup(K, N, bits, dtype):
    torch.manual_seed(K + N)
    q, lut = _words(bits, N, K // 32), torch.randn(N, 2 ** bits, device="cuda").to(dtype)
    want = F.dequant_lut(F.unpack_anyprec(q, bits), lut)
    assert torch.equal(ext.anyprec_dequant(q, lut, bits), want)
    apart = torch.empty(lut.numel() + 1, dtype=dtype, device="cuda")[1:].view(lut.shape)      # tables that start at an odd element
    apart.copy_(lut)
    assert torch.equal(ext.anyprec_dequant(q, apart, bits), want)


def _random_layer(fmt, bits, K, N, dtype, g):
    from decdec_amd import linear
    words = lambda *shape: torch.randint(-2 ** 31, 2 ** 31 - 1, shape, generator=g, device="cuda", dtype=torch.int32)
    randn = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    if fmt == "lutgemm":
        l = linear.LUTGEMMLinear(K, N, bits, 32 if K % 128 else 128, dtype=dtype)
        l.alpha.copy_(randn(*l.alpha.shape).abs() * 0.02)
        l.q_bias.copy_(randn(*l.q_bias.shape) * 0.002)
    else:
        l = (linear.APLinear if fmt == "anyprec" else linear.SQLLMLinear)(K, N, bits, dtype=dtype)
        l.lut.copy_(randn(*l.lut.shape).sort(1).values * 0.03)
    l.qweight.copy_(words(*l.qweight.shape))
    return l


# What a product's sums of shares take of its workspace: tiles of `mt` x 16 tokens and 128 outputs, of which the last are split and the first are not.
def _some_split(rows, dim, ff, mt):
    token_tiles = -(-rows // (16 * mt))
    groups = -(-2 * ff // 128)
    tiles = groups if token_tiles == 1 else -(-groups // 8) * 8 * token_tiles
    shares = _lib.load().decdec_quant_gemm_workspace_bytes(rows, dim, 2 * ff) / (16 * mt * 128 * 4)
    return tiles > 256 and shares > 0 and shares % (tiles - 256) == 0


# rows, width, feed-forward: one tile and less, remainders of every piece, split tiles, two token tiles, tiles of 256 tokens (300 and 500 rows of 12320; the latter in
# SqueezeLLM alone); and, by their 16-token tiles, whole tiles ahead of split ones: one token tile, two, in remainders, three (where a column has both)
@pytest.mark.parametrize("rows,dim,ff,mt", [(2, 256, 32, 0), (77, 512, 17920, 0), (17, 256, 224, 0), (77, 512, 1504, 0), (128, 1024, 4000, 0), (130, 256, 96, 0), (256, 320, 6176, 0),
                                            (100, 256, 10016, 0), (300, 1024, 12320, 0), (500, 1024, 12320, 0), (33, 96, 1184, 0),
                                            (77, 2048, 17920, 5), (61, 2080, 16416, 4), (200, 2048, 9056, 7), (256, 2048, 8224, 8), (300, 2048, 5664, 7)])
@pytest.mark.parametrize("fmt,bits,dtype", [("anyprec", 3, torch.bfloat16), ("lutgemm", 3, torch.float16), ("lutgemm", 4, torch.bfloat16), ("sqllm", 4, torch.float16),
                                            ("sqllm", 3, torch.bfloat16)])
def test_gate_and_up_in_one_product_that_gates(fmt, bits, dtype, rows, dim, ff, mt):
    """What is behind a block's attention: silu(gate) * up stored by the product itself (or by the sums of its shares) has the bits of the product, stored, and the
    activation of what is read back."""
    from decdec_amd import decode_ops
    from decdec_amd.linear import packed_layer
    assert mt == 0 or _some_split(rows, dim, ff, mt)
    g = torch.Generator(device="cuda").manual_seed(rows + ff)
    layers = [_random_layer(fmt, bits, K, N, dtype, g) for K, N in ((dim, dim), (dim, 2 * ff), (ff, dim))]
    x, y = (torch.randn(1, rows, dim, generator=g, device="cuda").to(dtype) for _ in range(2))
    norm = (1 + 0.1 * torch.randn(dim, generator=g, device="cuda")).to(dtype)
    with torch.no_grad():
        packed = [packed_layer(l, rows, dtype, 0) for l in layers]
        if rows > 256 and None in packed:                  # multiplied with expanded weights
            packed = [packed_layer(l, 2, dtype, 0) for l in layers]
        assert None not in packed
        h, out = torch.empty_like(x), torch.empty_like(x)
        scratch = torch.full((decode_ops.prompt_scratch_bytes(rows, dim, dim, ff),), 255, dtype=torch.uint8, device="cuda")
        decode_ops.prompt_back(x, y[0], norm, 1e-5, packed, h, out, scratch)

        def product(l, rows_in):
            table = l.alpha if fmt == "lutgemm" else l.lut
            if fmt == "lutgemm":
                return ext.lutgemm_gemm(rows_in, l.qweight, table, l.q_bias, bits, l.group_size)
            return (ext.anyprec_gemm if fmt == "anyprec" else ext.sqllm_gemm)(rows_in, l.qweight, table, bits)
        branch, want_h, n = product(layers[0], y[0]), torch.empty_like(x), torch.empty_like(x)
        decode_ops.add_rmsnorm(x, branch[None], norm, want_h, n, 1e-5)
        want = product(layers[2], decode_ops.silu_mul_rows(product(layers[1], n[0])))
        assert torch.equal(h, want_h)
        assert torch.equal(out[0], want)
