"""Mixer kernels against the plain oracle, each mechanism alone: in one portion, in portions of several sizes and token by
token, in float32 (tight) and bfloat16."""
import pytest
import torch

from decdec_amd import mixer_ops as M
from oracle import hybrid_oracle as O
import hybrid_cases as cases
from mixer_bench import Bench, close as _close, portions as _portions, rand as _rand

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]


# ---- rows --------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K,act", [(5, 3, 2), (64, 84, 0), (301, 200, 100), (4100, 96, 4100), (16400, 264, 8), (40, 2056, 1), (7, 1025, 3)])
def test_gemv_with_an_activation_on_its_first_rows(N, K, act, dtype):
    w, x, a = _rand(N, K, seed=N).to(dtype), _rand(K, seed=1).to(dtype), torch.tensor([0.7, -0.4]).to(dtype)
    out = torch.full((N,), 9.0, dtype=dtype, device="cuda")
    M.gemv(w.cuda(), x.cuda(), out, a.cuda() if act else None, act)
    y = w.double() @ x.double()
    y[:act] = O.xielu(y[:act], a[0].double(), a[1].double())
    _close(out, y, dtype)


# quarters of a row: fewer steps than waves, waves without a step, an odd number of steps, a ragged last step, an odd last row
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K", [(1, 8), (3, 512), (2, 1024), (5, 1536), (4, 2568), (9, 5128), (2, 14336)])
def test_gemv_at_the_edges_of_its_quarters(N, K, dtype):
    w, x = _rand(N, K, seed=N).to(dtype), _rand(K, seed=1).to(dtype)
    out = torch.full((N + 1,), 9.0, dtype=dtype, device="cuda")
    M.gemv(w.cuda(), x.cuda(), out[:N])
    # fp32 sums, one rounding to the storage type
    want, size = w.double() @ x.double(), w.double().abs() @ x.double().abs()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    assert ((out[:N].cpu().double() - want).abs() <= unit * want.abs() + 2.0 ** -20 * size).all() and float(out[N]) == 9.0


@pytest.mark.parametrize("dtype", DTYPES)
def test_gemv_of_extremes(dtype):
    """Numbers below the normal ones count, infinities stay, and nothing else changes beside them."""
    N, K = 6, 2048
    w, x = torch.zeros(N, K), torch.ones(K)
    x[:8] = 2.0 ** 126
    w[0, :8], w[1, 9], w[2, 10], w[3, 11] = 2.0 ** -130, float("inf"), -float("inf"), float("nan")
    w[4, 12], w[5, 0::2], w[5, 1::2] = 2.0 ** -120, 2.0 ** -2, -2.0 ** -2
    w[5, -1] = 1.75
    out = torch.empty(N, dtype=dtype, device="cuda")
    M.gemv(w.to(dtype).cuda(), x.to(dtype).cuda(), out)
    got = out.cpu().float().tolist()
    assert got[0] == 0.5 and got[1] == float("inf") and got[2] == -float("inf") and got[3] != got[3]
    assert got[4] == 2.0 ** -120 and got[5] == 2.0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K", [(5, 3), (301, 200), (4100, 96)])
def test_gemv_with_gelu_and_a_scale(N, K, dtype):
    w, x = _rand(N, K, seed=N).to(dtype), _rand(K, seed=1).to(dtype)
    y = w.double() @ x.double()
    out = torch.empty(N, dtype=dtype, device="cuda")
    M.gemv(w.cuda(), x.cuda(), out, None, N, M.ACT_GELU_TANH)
    _close(out, O.gelu_tanh(y), dtype)
    M.gemv(w.cuda(), x.cuda(), out, scale=0.3)
    _close(out, 0.3 * y, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K,first", [(1, 8, 0), (5, 3, 0), (301, 200, 0), (2048, 7168, 0), (33, 96, 1)])
def test_gemv_with_residual_and_norm_is_both_in_turn(N, K, first, dtype):
    """Bit for bit; first = 1: an input that starts between two pieces of 16 bytes."""
    w, inp = _rand(N, K, seed=N).to(dtype).cuda(), _rand(K + 1, seed=1).to(dtype).cuda()[first:first + K]
    x, norm = _rand(1, N, seed=2).cuda(), tuple(t.to(dtype).cuda() for t in (torch.tensor(0.7), _rand(N, seed=3), _rand(N, seed=4)))
    y, want, got = (torch.empty(1, N, dtype=dtype, device="cuda") for _ in range(3))
    want_x, got_x = x.clone(), x.clone()
    M.gemv(w, inp, y)
    M.residual_tanh(want_x, y, norm, want)
    M.gemv_residual_tanh(w, inp, got_x, norm, got)
    assert torch.equal(got_x, want_x) and torch.equal(got, want)
    with pytest.raises(RuntimeError):
        M.gemv_residual_tanh(w, inp, got_x, norm, inp)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,dim", [(1, 84), (3, 33), (4, 4096), (2, 7001)])
def test_residual_and_embedding_behind_a_dynamic_tanh(rows, dim, dtype):
    x, y = _rand(rows, dim, seed=1, scale=3.0), _rand(rows, dim, seed=2).to(dtype)
    x[0, :7] = torch.tensor([0.0, 1e-6, -1e-4, 1e-2, 40.0, -40.0, 300.0])     # near zero and far past saturation
    a, w, b = torch.tensor(0.7).to(dtype), _rand(dim, seed=5).to(dtype), _rand(dim, seed=6).to(dtype)
    norm = tuple(t.cuda() for t in (a, w, b))
    want = lambda v: O.dynamic_tanh(v, a.double(), w.double(), b.double())
    xd, out = x.cuda(), torch.empty(rows, dim, dtype=dtype, device="cuda")
    M.residual_tanh(xd, None, norm, out)
    assert torch.equal(xd.cpu(), x)
    _close(out, want(x.double()), dtype)
    M.residual_tanh(xd, y.cuda(), norm, out)
    assert torch.equal(xd.cpu(), x + y.float())            # the residual stream is float32 whatever the storage type
    _close(out, want(x.double() + y.double()), dtype)
    no_bias = (norm[0], norm[1], torch.zeros_like(norm[2]))
    small = (_rand(rows, dim, seed=7) * 1e-4).cuda()       # tanh keeps its relative accuracy there
    M.residual_tanh(small, None, no_bias, out)
    _close(out, torch.tanh(a.double() * small.double().cpu()) * w.double(), dtype)
    table, toks = _rand(50, dim, seed=8).to(dtype).cuda(), torch.tensor([3, 49, 0, 3][:rows], device="cuda")
    M.embed(table, toks, xd, out, norm)
    assert torch.equal(xd, table[toks].float())
    _close(out, want(table[toks].double().cpu()), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,ld", [(52, 60), (7, 9), (5000, 5000)])
def test_gelu_rows(n, ld, dtype):
    inp = _rand(3, ld, seed=4, scale=3.0).to(dtype).cuda()
    want = O.gelu_tanh(inp[:, :n].double().cpu())
    out = inp if n == ld else torch.empty(3, n, dtype=dtype, device="cuda")   # in place where the rows are whole
    M.activation(inp, n, None, out, M.ACT_GELU_TANH)
    _close(out, want, dtype)


# a workgroup a piece of a row, some pieces and a whole row (xIELU in bf16); rows that end inside a piece, and of single elements
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,n", [(300, 9004), (1100, 9004), (2100, 9004), (2100, 4097)])
def test_activation_of_many_rows(rows, n, dtype):
    inp, a = _rand(rows, n, seed=rows, scale=2.0).to(dtype).cuda(), torch.tensor([-0.3, 1.2]).to(dtype).cuda()
    out = torch.empty_like(inp)
    M.activation(inp, n, a, out)
    _close(out, O.xielu(inp.double(), a[0].double(), a[1].double()), dtype)
    M.activation(inp, n, None, out, M.ACT_GELU_TANH)
    _close(out, O.gelu_tanh(inp.double()), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("groups,n", [(3, 36), (3, 128), (2, 256), (2, 201), (2, 1028), (1, 1030)])
@pytest.mark.parametrize("at,wide", [(0, 0), (8, 16), (3, 5)])
def test_group_norm_gate_into_columns_with_a_scale(groups, n, at, wide, dtype):
    o, g, w = _rand(3, groups * n, seed=1).cuda(), _rand(3, groups * n, seed=2).to(dtype).cuda(), _rand(n, seed=3).to(dtype).cuda()
    buf = torch.full((3, groups * n + wide), 7.0, dtype=dtype, device="cuda")
    out = buf[:, at:at + groups * n]
    M.group_norm_gate(o, g, groups * n, w, out, groups, 0.01, M.GATE_SILU, 0.3)
    want = 0.3 * O.rms_norm(o.double().view(3, groups, n), w.double(), 0.01).view(3, -1) * O.silu(g.double())
    _close(out, want, dtype)
    assert float((buf[:, :at] - 7).abs().sum() + (buf[:, at + groups * n:] - 7).abs().sum()) == 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,dim,gate,final", [(1, 84, True, True), (3, 84, True, False), (2, 33, True, True), (4, 4096, False, True),
                                                 (2, 7000, True, True), (1, 16384, True, False), (2, 20000, True, True)])
def test_gated_residual(rows, dim, gate, final, dtype):
    eps = 1e-3
    x, y = _rand(rows, dim, seed=1, scale=3.0), _rand(rows, dim, seed=2, scale=0.05).to(dtype)
    g, b, w, fw = _rand(rows, dim + 12, seed=3).to(dtype), _rand(dim, seed=4).to(dtype), _rand(dim, seed=5).to(dtype), _rand(dim, seed=6).to(dtype)
    xd, gd = x.cuda(), g.cuda()
    xe, fo = (torch.empty(rows, dim, dtype=dtype, device="cuda") for _ in range(2))
    M.gated_residual(xd, y.cuda(), gd[:, 8:] if gate else None, dim + 12, b.cuda() if gate else None, w.cuda(), xe, eps,
                     fw.cuda() if final else None, fo if final else None)
    y = y.double() * (O.sigmoid(g[:, 8:8 + dim].double() + b.double()) if gate else 1.0)
    want = x.double() + O.rms_norm(y, w.double(), eps)
    _close(xd, want, torch.float32)                     # the residual stream is float32 whatever the storage type
    _close(xe, want, dtype)
    if final:
        _close(fo, O.rms_norm(want, fw.double(), eps), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed_norm_and_activation_rows(dtype):
    table = _rand(50, 21, seed=1).to(dtype).cuda()
    toks = torch.tensor([3, 49, 0, 3], device="cuda")
    x, xe = torch.empty(4, 21, device="cuda"), torch.empty(4, 21, dtype=dtype, device="cuda")
    M.embed(table, toks, x, xe)
    assert torch.equal(x, table[toks].float()) and torch.equal(xe, table[toks])
    M.embed(table, torch.tensor([50, -1, 2, 1], device="cuda"), x, None)          # ids outside the table read row 0
    assert torch.equal(x[:2], table[[0, 0]].float())
    for rows, dim in ((3, 21), (2, 5000)):
        v, w = _rand(rows, dim, seed=2).cuda(), _rand(dim, seed=3).to(dtype).cuda()
        out = torch.empty(rows, dim, dtype=dtype, device="cuda")
        M.rmsnorm(v, w, out, 0.1)
        _close(out, O.rms_norm(v.double(), w.double(), 0.1), dtype)
    for n, ld in ((52, 60), (7, 9), (5000, 5008)):
        inp, a = _rand(3, ld, seed=4, scale=2.0).to(dtype).cuda(), torch.tensor([-0.3, 1.2]).to(dtype).cuda()
        out = torch.empty(3, n, dtype=dtype, device="cuda")
        M.activation(inp, n, a, out)
        _close(out, O.xielu(inp[:, :n].double(), a[0].double(), a[1].double()), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("groups,n,kind", [(1, 140, M.GATE_SIGMOID), (3, 36, M.GATE_SILU), (2, 2048, M.GATE_SILU), (3, 128, M.GATE_SILU),
                                           (2, 256, M.GATE_SIGMOID), (2, 201, M.GATE_SILU), (1, 1030, M.GATE_SIGMOID)])
@pytest.mark.parametrize("off,pad", [(2, 5), (8, 16)])
def test_group_norm_gate(groups, n, kind, off, pad, dtype):
    o, g, w = _rand(3, groups * n, seed=1).cuda(), _rand(3, groups * n + pad, seed=2).to(dtype).cuda(), _rand(n, seed=3).to(dtype).cuda()
    out = torch.empty(3, groups * n, dtype=dtype, device="cuda")
    M.group_norm_gate(o, g[:, off:], groups * n + pad, w, out, groups, 0.01, kind)
    z = g[:, off:off + groups * n].double()
    want = O.rms_norm(o.double().view(3, groups, n), w.double(), 0.01).view(3, -1) * (O.silu(z) if kind == M.GATE_SILU else O.sigmoid(z))
    _close(out, want, dtype)


# ---- mixers ------------------------------------------------------------------------------------------------
RECURRENCES = [("lightning", cases.lightning(3, 32, 32)), ("lightning", cases.lightning(5, 12, 28, [0.0, 0.3, 0.95, 0.9999, 1.0])),
               ("lightning", cases.lightning(2, 128, 128)), ("lightning", cases.lightning(1, 200, 72, [0.98])), ("lightning", cases.lightning(2, 1, 1)),
               ("delta", cases.delta(4, 2, 48, 64, 4)), ("delta", cases.delta(3, 3, 20, 36, 3)), ("delta", cases.delta(4, 2, 128, 128, 4)),
               ("delta", cases.delta(2, 2, 64, 16, 1)), ("delta", cases.delta(6, 2, 9, 130, 2)), ("delta", cases.delta(1, 1, 256, 256, 7)),
               ("delta", cases.delta(2, 1, 16, 300, 5)),
               ("gated_linear", cases.gated_linear(3, 32, 32, 16.0)), ("gated_linear", cases.gated_linear(5, 12, 28, 1.0)),
               ("gated_linear", cases.gated_linear(2, 128, 128, 4.0)), ("gated_linear", cases.gated_linear(1, 200, 72, 0.5)),
               ("gated_linear", cases.gated_linear(2, 1, 1, 2.0)), ("gated_linear", cases.gated_linear(2, 48, 2000, 8.0)),
               ("channel_delta", cases.delta(4, 2, 48, 64, 4)), ("channel_delta", cases.delta(3, 3, 20, 36, 3)),
               ("channel_delta", cases.delta(4, 2, 128, 128, 4)), ("channel_delta", cases.delta(2, 2, 64, 16, 1)),
               ("channel_delta", cases.delta(6, 2, 9, 130, 2)), ("channel_delta", cases.delta(1, 1, 256, 256, 7)),
               ("channel_delta", cases.delta(2, 1, 16, 300, 9)), ("channel_delta", cases.delta(1, 1, 30, 1100, 4))]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind,m", RECURRENCES)
def test_recurrence_in_portions_and_token_by_token(kind, m, dtype):
    T = 150
    b = Bench(kind, m, dtype, T)
    want = b.want()
    for sizes in ((T,), (2,), (3, 64, 1, 2), (65, 63, 5), (1,), (130, 1)):
        # the state of the sequence before is left in place: position 0 starts afresh
        _close(b.run(_portions(T, *sizes)), want, dtype, (kind, m, sizes), factor=4.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D,V", [(64, 16), (63, 15), (65, 17), (192, 32), (256, 16)])
@pytest.mark.parametrize("kind", ["lightning", "gated_linear", "delta", "channel_delta"])
def test_states_at_the_edges_of_their_blocks(kind, D, V, dtype):
    """Blocks of 64 rows and 16 columns of the state, chunks of 64 tokens: one more and one less of each."""
    m = cases.lightning(2, D, V) if kind == "lightning" else (cases.gated_linear(2, D, V, 0.35) if kind == "gated_linear" else cases.delta(2, 1, D, V, 3))
    T = 194
    b = Bench(kind, m, dtype, T)
    want = b.want()
    for sizes in ((T,), (64, 65, 63), (128, 1)):
        _close(b.run(_portions(T, *sizes)), want, dtype, (kind, m, sizes), factor=4.0)


@pytest.mark.parametrize("dtype", DTYPES)
def test_delta_rule_with_decays_that_forget_at_once_and_never(dtype):
    def edit(b):
        b.w["A_log"] = torch.tensor([5.0, -12.0, 2.0]).to(torch.bfloat16)
        b.w["dt_bias"] = torch.tensor([4.0, -6.0, 1.0]).to(torch.bfloat16)
    b = Bench("delta", cases.delta(3, 1, 24, 24, 4), dtype, 140, edit=edit)
    for sizes in ((140,), (37,), (1,)):
        _close(b.run(_portions(140, *sizes)), b.want(), dtype, sizes, factor=4.0)


@pytest.mark.parametrize("kind", ["delta", "channel_delta"])
def test_convolution_sees_exactly_its_taps_across_a_cut(kind):
    """One token's input is changed: the read-outs of a head without memory differ for `taps` tokens from there on, no
    more and no fewer, wherever the portions are cut."""
    taps, T = 4, 40

    def edit(b):                                           # a decay of e^-150: nothing but the convolution reaches back
        b.w["A_log"], b.w["dt_bias"] = torch.tensor([5.0]).to(torch.bfloat16), torch.full_like(b.w["dt_bias"], 4.0)
        a = "a" if kind == "delta" else "a1"
        b.w[a] = torch.zeros_like(b.w[a])
    b = Bench(kind, cases.delta(1, 1, 16, 16, taps), torch.float32, T, edit=edit)
    for sizes in ((T,), (1,), (2,), (7, 1)):
        base = b.run(_portions(T, *sizes))
        keep = b.proj.clone()
        for at in (0, 6, 7, 13):
            b.proj[at, :48] += 1.0                         # q, k and v of one token
            moved = (b.run(_portions(T, *sizes)) - base).abs().amax(1) > 1e-4
            assert moved.nonzero().view(-1).tolist() == list(range(at, at + taps)), (sizes, at)
            b.proj.copy_(keep)


def _channel_extremes(kind, H, D):
    """Per channel: forgetting at once, never, and everything between, side by side in a head."""
    def edit(b):
        g = torch.Generator().manual_seed(3)
        bias = torch.randn(H * D, generator=g) * 3.0
        bias[::5], bias[1::5] = -30.0, 30.0
        b.w["a2.b" if kind == "gated_linear" else "dt_bias"] = bias.to(torch.bfloat16)
        if kind == "channel_delta":
            b.w["A_log"] = torch.tensor([4.0, -9.0, 1.0][:H]).to(torch.bfloat16)
    return edit


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["gated_linear", "channel_delta"])
def test_channel_decays_that_forget_at_once_and_never(kind, dtype):
    m = cases.gated_linear(3, 40, 24, 0.25) if kind == "gated_linear" else cases.delta(3, 1, 40, 24, 4)
    b = Bench(kind, m, dtype, 200, edit=_channel_extremes(kind, 3, 40))
    want = b.want()
    for sizes in ((200,), (37,), (1,)):
        _close(b.run(_portions(200, *sizes)), want, dtype, (kind, sizes), factor=4.0)


@pytest.mark.parametrize("kind", ["gated_linear", "channel_delta"])
def test_tokens_that_forget_everything_between_tokens_that_keep(kind):
    """Decays near one among decays of e^-160 and less: what is written after a token that forgets lasts, whatever the sums hold."""
    T, D, V = 140, 24, 16

    def edit(b):
        z = torch.full((T,), -6.0)
        z[[5, 6, 7, 8, 20, 63, 64, 100]] = 60.0
        b.h[:, 0] = (z if kind == "channel_delta" else -z).to(torch.bfloat16)
        for n in ("q", "k", "v", "b", "g", "g1"):
            if n in b.w:
                b.w[n][:, 0] = 0
        b.w["a1"].zero_(), b.w["a2"].zero_()
        b.w["a1"][0, 0] = 1
        b.w["a2"][:, 0] = 1
        if kind == "channel_delta":
            b.w["A_log"][:] = 1.0
        b.w["dt_bias" if kind == "channel_delta" else "a2.b"].mul_(0.1)
    m = cases.gated_linear(1, D, V, 0.35) if kind == "gated_linear" else cases.delta(1, 1, D, V, 2)
    b = Bench(kind, m, torch.float32, T, edit=edit)
    want = b.want()
    for sizes in ((T,), (1,), (50, 3)):
        _close(b.run(_portions(T, *sizes)), want, torch.float32, sizes, factor=2.0)


@pytest.mark.parametrize("kind", ["gated_linear", "channel_delta"])
def test_every_key_channel_has_its_own_decay(kind):
    """A head whose channels all forget at once but one: what a token wrote comes back through that channel alone, from any
    distance and over any cut."""
    T, D, V, keep = 150, 24, 16, 7
    m = cases.gated_linear(1, D, V, 1.0) if kind == "gated_linear" else cases.delta(1, 1, D, V, 1)

    def edit(b):
        forget = -60.0 if kind == "gated_linear" else 60.0                     # sigmoid(-60), or exp(-e softplus(60))
        bias = torch.full((D,), forget)
        bias[keep] = -forget
        b.w["a2.b" if kind == "gated_linear" else "dt_bias"] = bias.to(torch.bfloat16)
        b.w["a1"] = torch.zeros_like(b.w["a1"])
        if kind == "channel_delta":
            b.w["A_log"] = torch.tensor([1.0]).to(torch.bfloat16)
    b = Bench(kind, m, torch.float32, T, edit=edit)
    want = b.want()
    for sizes in ((T,), (1,), (50, 3), (65,)):
        base = b.run(_portions(T, *sizes))
        _close(base, want, torch.float32, sizes, factor=4.0)
    k = b.mixer.params.off_k
    saved = b.proj.clone()
    b.proj[3, k + keep] += 3.0                                                 # the lasting channel of an early key
    far = (b.run([T]) - base).abs().amax(1)
    assert float(far[100:].max()) > 1e-3 and float(far[:3].max()) < 1e-6
    if kind == "gated_linear":                                                 # (unit vectors couple the channels)
        b.proj.copy_(saved)
        b.proj[3, k + keep + 1] += 3.0
        moved = (b.run([T]) - base).abs().amax(1) > 1e-5
        assert moved.nonzero().view(-1).tolist() == [3]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rank", [1, 7, 64, 200, 1024])
def test_low_rank_maps_of_any_rank(rank, dtype):
    def edit(b):
        g, H, D, V = torch.Generator().manual_seed(rank), 2, 16, 24
        put = lambda n, *s: b.w.__setitem__(n, (torch.randn(*s, generator=g) * 1.5 / s[1] ** 0.5).to(torch.bfloat16))
        put("a1", rank, 40), put("a2", H * D, rank), put("g1", rank, 40), put("g2", H * V, rank)
    b = Bench("channel_delta", cases.delta(2, 1, 16, 24, 4), dtype, 70, edit=edit)
    want = b.want()
    for sizes in ((70,), (1,)):
        _close(b.run(_portions(70, *sizes)), want, dtype, (rank, sizes), factor=4.0)


LATENTS = [cases.latent(3, 64, 32, 96, 80, scaling=cases.YARN), cases.latent(3, 22, 10, 18, 30, base=500.0), cases.latent(17, 16, 8, 24, 48, scale=0.4),
           cases.latent(2, 128, 64, 128, 512, base=10000.0), cases.latent(1, 200, 56, 200, 96), cases.latent(2, 32, 16, 40, 72, dims=8),
           cases.latent(1, 2, 2, 1, 1), cases.latent(2, 96, 64, 256, 136)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m", LATENTS)
def test_latent_attention_in_portions_and_token_by_token(m, dtype):
    T = 150
    b = Bench("latent_attention", m, dtype, T)
    want = b.want()
    for sizes in ((T,), (2,), (3, 64, 1, 2), (65, 63, 5), (1,), (130, 1)):
        _close(b.run(_portions(T, *sizes)), want, dtype, (m, sizes), factor=2.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("scale", [-0.4, 0.0])
@pytest.mark.parametrize("dim,rot", [(24, 8), (128, 64)])
def test_latent_attention_with_a_scale_that_is_not_positive(dim, rot, scale, dtype):
    """The tiled kernel takes its maximum before it scales: a negative scale turns the order around, and of none all visible keys
    weigh the same.  Keys that fill their tile, and keys that leave part of it empty."""
    T, m = 150, cases.latent(2, dim, rot, 40, 48, scale=scale)
    b = Bench("latent_attention", m, dtype, T)
    want = b.want()
    for sizes in ((T,), (65, 63, 5)):
        _close(b.run(_portions(T, *sizes)), want, dtype, (m, sizes), factor=2.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("max_seq", [700, 8000])
def test_latent_attention_finds_one_key_at_every_tile_edge(dtype, max_seq):
    """A query is made to point at one key: its read-out is that token's value, wherever the key lies relative to the tiles
    of 64 keys and to the shares of the one-token kernel's workgroups."""
    T, m = 700, cases.latent(2, 32, 8, 32, 48, base=1e6, scale=1.0)
    b = Bench("latent_attention", m, dtype, T, max_seq=max_seq)
    H, D, R, V, C = 2, 32, 8, 32, 48
    c = O.rms_norm(b.proj[:, 80:80 + C].double().cpu(), b.w["dkv.norm"].double(), b.eps)
    kn = (c @ b.w["uk"].double().T).view(T, H, D)
    v = (c @ b.w["uv"].double().T).view(T, H * V)
    b.run([T - 1])
    tried = 0
    for key in (0, 1, 62, 63, 64, 65, 127, 128, 319, 320, 511, 512, 575, 576, 640, 697, 698):
        q = torch.zeros(H, D + R, dtype=torch.float64)
        for h in range(H):
            others = torch.cat((kn[:key, h], kn[key + 1:, h]))
            q[h, :D] = kn[key, h] * 60.0 / float(kn[key, h] @ kn[key, h] - (others @ kn[key, h]).max()).__abs__()
        b.proj[T - 1, :80] = q.view(-1).to(dtype)
        scores = torch.stack([kn[:, h] @ b.proj[T - 1].double().cpu()[:80].view(H, D + R)[h, :D] for h in range(H)])
        if (scores.argmax(1) != key).any():
            continue                                       # a longer key in the same direction wins
        tried += 1
        one = b.run([1], T - 1)
        for name, got in (("one token", one[0]), ("portion", b.run([3], T - 3)[2])):
            e = torch.exp(scores - scores.amax(1, keepdim=True))
            want = torch.cat([(e[h] / (e[h].sum() + torch.exp(b.w["sink"][h].double() - scores[h].max()))) @ v.view(T, H, V)[:, h] for h in range(H)])
            _close(got, want, dtype, (name, key), factor=3.0)
    assert tried >= 14


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("max_seq", [4170, 9000])
def test_latent_step_around_64_tiles(max_seq, dtype):
    """4096 keys and a few more, a tile of 64 a workgroup."""
    T = 4164
    b = Bench("latent_attention", cases.latent(2, 16, 8, 16, 24), dtype, T, max_seq=max_seq)
    want = b.want()
    for at in (4094, 4158):                                # 4095 .. 4098 and 4159 .. 4164 keys
        b.run([at])
        n = min(6, T - at)
        _close(b.run([1] * n, at), want[at:at + n], dtype, at, factor=2.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,tiles", [(2, 104), (31, 104), (32, 64)])
def test_latent_step_around_the_length_from_which_shares_are_two_tiles(heads, tiles, dtype):
    """In bf16 as many tiles go to a workgroup each, more in twos, the last one alone; in 32 bits one each.  Against a prompt of as many tokens."""
    T = 64 * tiles + 68
    b = Bench("latent_attention", cases.latent(heads, 16, 8, 16, 24), dtype, T, max_seq=9000)
    want = b.run([T]).clone()
    for at in (64 * tiles - 2, 64 * tiles + 62):
        b.run([at])
        _close(b.run([1] * 6, at), want[at:at + 6], dtype, at, factor=2.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sink", [-30.0, 0.0, 12.0])
def test_sink_counts_once_whatever_the_number_of_workgroups(sink, dtype):
    def edit(b):
        b.w["sink"] = torch.tensor([sink, sink / 2]).to(torch.bfloat16)
    b = Bench("latent_attention", cases.latent(2, 16, 8, 16, 24), dtype, 520, edit=edit)
    want = b.want()
    _close(b.run([520]), want, dtype, factor=2.0)
    _close(b.run([1] * 5), want[:5], dtype, factor=2.0)                 # the first tokens
    b.run([515])
    _close(b.run([1] * 5, 515), want[515:], dtype, factor=2.0)


def test_no_key_after_the_query_and_every_key_up_to_it():
    """The last visible key is the query's own: changing a later token's input changes nothing, changing its own does."""
    T = 140
    b = Bench("latent_attention", cases.latent(2, 16, 8, 16, 24), torch.float32, T)
    base = b.run([T])
    for at in (0, 1, 63, 64, 127, 128, 139):
        keep = b.proj.clone()
        b.proj[at, 48:48 + 32] += 2.0                                    # latent and rotated key of one token
        for sizes in ((T,), (70,), (1,)):
            diff = (b.run(_portions(T, *sizes)) - base).abs().amax(1)
            assert float(diff[:at].max() if at else 0.0) < 1e-5 and float(diff[at]) > 1e-4, (at, sizes)
        b.proj.copy_(keep)


def test_a_cache_of_a_longer_sequence_before_is_not_seen():
    m = cases.latent(2, 16, 8, 16, 24)
    b = Bench("latent_attention", m, torch.float32, 300)
    b.run([300])
    short = Bench("latent_attention", m, torch.float32, 70, seed=9, max_seq=300)
    short.state = b.state                                                # full of the other sequence's rows
    want = short.want()
    _close(short.run([69]), want[:69], torch.float32)
    _close(short.run([1], 69), want[69:], torch.float32)


# ---- products of several rows --------------------------------------------------------------------------------
# tiles of 16 tokens (every number of them, two and three groups), of 128 outputs, steps of 32 and 64 elements (one, odd, ragged),
# ranges of K, outputs that are no multiple of four, rows that are apart
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,N,K", [(1, 1, 8), (16, 128, 32), (17, 130, 64), (40, 257, 96), (64, 64, 1000), (80, 132, 2056), (96, 128, 72),
                                      (112, 31, 4096), (128, 256, 136), (129, 300, 520), (300, 384, 264), (777, 129, 1032)])
def test_product_of_rows(rows, N, K, dtype):
    wide = _rand(rows, K + 24, seed=rows).to(dtype).cuda()
    x, w = wide[:, 16:16 + K], _rand(N, K, seed=1).to(dtype).cuda()
    got = M.row_gemm(x, w).double()
    want, size = x.double() @ w.double().T.contiguous(), x.double().abs() @ w.double().abs().T.contiguous()
    # one rounding to the storage type; every matrix instruction (32 channels; six products of them in float32) may round its sum,
    # at most the sum of all terms' sizes, by a unit, and three products of the nine, 2^-24 together, are left out
    unit, passes = (2.0 ** -8, 1) if dtype == torch.bfloat16 else (2.0 ** -24, 6)
    assert ((got - want).abs() <= unit * want.abs() + (passes * ((K + 31) // 32) + 1) * 2.0 ** -23 * size).all()


def test_float_product_is_as_exact_as_a_float_product():
    """Sums whose terms cancel, and factors of very different sizes: no further from 64 bits than torch's float32 product."""
    g = torch.Generator().manual_seed(0)
    x = torch.randn(192, 2048, generator=g) * torch.exp(2 * torch.randn(192, 1, generator=g))
    w = torch.randn(384, 2048, generator=g) * torch.exp(torch.randn(384, 2048, generator=g))
    w[:, 1024:] = -w[:, :1024] * (1 + 2.0 ** -12 * torch.randn(384, 1024, generator=g))
    x[:, 1024:] = x[:, :1024]
    want = x.double() @ w.double().T
    off = lambda y: float((y.cpu().double() - want).norm() / want.norm())
    assert off(M.row_gemm(x.cuda(), w.cuda())) <= 1.1 * off(x.cuda() @ w.cuda().T)


@pytest.mark.parametrize("small", ["x", "w", "some rows of both"])
def test_float_product_of_small_numbers(small):
    """Rows whose trailing bits lie below what bf16 can hold."""
    g = torch.Generator().manual_seed(3)
    num = lambda *s: (torch.rand(*s, generator=g) * 0.5 + 0.5) * (torch.randint(0, 2, s, generator=g) * 2 - 1)
    x, w = num(192, 512), num(256, 512)
    if small == "x":
        x *= 2.0 ** -120
    elif small == "w":
        w *= 2.0 ** -118
    else:
        x[5::7] *= 2.0 ** -122
        w[3::50] *= 2.0 ** -4
    want = x.double() @ w.double().T
    got = M.row_gemm(x.cuda(), w.cuda()).cpu().double()
    # each output within the rounding of its sums: 512 terms, 2^-24 each of at most the sum of sizes, as a random walk of 128 steps
    size = x.double().abs() @ w.double().abs().T
    assert ((got - want).abs() <= 2.0 ** -19 * size / 512 ** 0.5 + 2.0 ** -140).all()


def test_float_product_of_extremes():
    """Infinities, NaN and numbers that bf16 cannot hold stay what they are."""
    x, w = torch.zeros(160, 64), torch.zeros(128, 64)
    x[0, 0], x[1, 1], x[2, 2], x[3, 3], x[4, 4] = float("inf"), float("nan"), 3.4e38, 1e-30, -float("inf")
    w[torch.arange(64), torch.arange(64)] = 1.0
    w[70, 0], w[71, 4] = 2.0, 3.0
    got = M.row_gemm(x.cuda(), w.cuda()).cpu()
    assert got[0, 0] == float("inf") and got[0, 70] == float("inf") and got[4, 71] == -float("inf") and torch.isnan(got[1, 1])
    assert got[2, 2] == x[2, 2] and got[3, 3] == x[3, 3] and not got[5:].any()


# float32 on the fp16 units: every number of tiles, one and several ranges of K, an odd and an even number of steps of a range and none for one
# of its halves, outputs that are no multiple of four, of 64 or of 256, tokens one short of and one past a block
def _in_two_pieces(rows, N, K):
    """Ranges of K of a product on fp16 pieces, 0 if it does not run on them."""
    return M._lib.load_mixers().decdec_mix_row_gemm_pieces(0, rows, N, K, K)


def _within_two_pieces(got, x, w):
    """Per product the two roundings of 2^-23 and what is left out, 2^-22; three additions of 32 channels' products, and those of the two halves
    and the ranges; weights below 2^-33 of the largest of a row's sample (at most that of the row) are cut off."""
    K, x, w = x.shape[1], x.double(), w.double()
    want, size = x @ w.T.contiguous(), x.abs() @ w.abs().T.contiguous()
    cut = 2.0 ** -33 * x.abs().sum(1, keepdim=True) * w.abs().amax(1)
    return ((got.double() - want).abs() <= 2.0 ** -24 * want.abs() + (4 + 3 * (K // 32) + 18) * 2.0 ** -23 * size + cut).all()


@pytest.mark.parametrize("rows,N,K", [(160, 8448, 2048), (161, 8451, 2080), (191, 4097, 4128), (225, 8193, 1056), (255, 2049, 7168), (448, 2304, 2080),
                                      (2000, 1793, 544), (777, 14336, 512), (777, 2047, 2048), (800, 4300, 1568), (1001, 1793, 640)])
def test_float_product_in_two_pieces(rows, N, K):
    assert _in_two_pieces(rows, N, K)
    wide = _rand(rows, K + 24, seed=rows).cuda()
    x, w = wide[:, 16:16 + K], _rand(N, K, seed=1).cuda()
    got = M.row_gemm(x, w)
    assert _within_two_pieces(got, x, w)
    want = x.double() @ w.double().T.contiguous()
    off = lambda y: float((y.double() - want).norm() / want.norm())
    assert off(got) <= off(x @ w.T)


# one range and several; four, five, six and seven tiles of 16 tokens a workgroup
@pytest.mark.parametrize("rows,N,K,ranges", [(800, 4300, 1568, 1), (160, 8448, 2048, 3), (161, 8451, 2080, 3), (777, 2304, 2048, 4)])
@pytest.mark.parametrize("case", ["outlier in w", "sample of zeros", "rows of zeros", "outlier in x", "tiny row of x", "tiny row of w", "infinite", "nan"])
def test_float_product_that_two_pieces_do_not_hold(case, rows, N, K, ranges):
    """Rows that no scale fits, beside rows that have one."""
    assert _in_two_pieces(rows, N, K) == ranges
    x, w = _rand(rows, K, seed=5).cuda(), _rand(N, K, seed=6).cuda()
    if case == "outlier in w":
        w[300, 37] = 3e6                                   # 32 .. 63 are in no sample of the first rows
        w[2303, 1] = -1e30
    elif case == "sample of zeros":
        w[7] = 0
        w[7, 40:50] = 3.0
        w[700, :] = 0
        w[700, 1023] = 1e-20
    elif case == "rows of zeros":
        w[5:900] = 0
        x[17] = 0
    elif case == "outlier in x":
        x[33, 900] = 1e25
    elif case == "tiny row of x":
        x[44] *= 2.0 ** -120
    elif case == "tiny row of w":
        w[55] *= 2.0 ** -120
    elif case == "infinite":
        x[3, 3], w[1000, 77] = float("inf"), -float("inf")
    else:
        x[3, 3], w[1000, 77] = float("nan"), float("nan")
    got = M.row_gemm(x, w)
    if case in ("infinite", "nan"):
        want = x.double() @ w.double().T.contiguous()
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isposinf(got), torch.isposinf(want))
        ok = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), ok)
        x[3, 3] = w[1000, 77] = 0
        again = x.double() @ w.double().T.contiguous()
        assert ((got - again).abs()[ok] <= 2.0 ** -12 * again.abs().max()).all()
    else:
        # an underflow of a float sum: half the smallest number a term
        size = x.double().abs() @ w.double().abs().T.contiguous()
        far = (got.double() - x.double() @ w.double().T.contiguous()).abs() > (3 * K // 32 + 24) * 2.0 ** -23 * size + 2.0 ** -140
        assert not far.any()


# four, five, six and seven tiles of 16 tokens a workgroup
@pytest.mark.parametrize("rows,N,K,ranges", [(800, 4300, 1568, 1), (160, 8448, 2048, 3), (161, 8451, 2080, 3), (777, 2047, 2048, 4)])
@pytest.mark.parametrize("case", ["opposed 1", "opposed 2", "opposed 2.5", "opposed 3", "w 300", "w 3e3", "w 1e4", "w 1e5", "w 3e6", "x 1e4", "x 1e5", "x 1e6", "x 1e25",
                                  "cancelling"])
def test_float_product_of_numbers_far_apart(case, rows, N, K, ranges):
    """Weights spread by channel and activations the other way, a channel far above the others in one of them that is zero in the other, sums
    whose terms cancel: no further from 64 bits than torch's float32 product, where small numbers of a row are what counts."""
    assert _in_two_pieces(rows, N, K) == ranges
    x, w = _rand(rows, K, seed=5).cuda(), _rand(N, K, seed=6).cuda()
    kind, _, size = case.partition(" ")
    if kind == "opposed":
        spread = torch.exp(float(size) * _rand(K, seed=7).cuda())
        x, w = x * spread, w / spread
    elif kind == "cancelling":
        h = K // 2
        w[:, h:], x[:, h:] = -w[:, :h] * (1 + 2.0 ** -12 * _rand(N, h, seed=8).cuda()), x[:, :h]
    else:                                                  # channel 0 is in the sample of some weight rows
        (w if kind == "w" else x)[:, 0], (x if kind == "w" else w)[:, 0] = float(size), 0.0
    want = x.double() @ w.double().T.contiguous()
    off = lambda y: float((y.double() - want).norm() / want.norm())
    assert off(M.row_gemm(x, w)) <= off(x @ w.T)


@pytest.mark.parametrize("rows,N,K,ranges", [(777, 2047, 2048, 4), (800, 4300, 1568, 1)])
def test_float_product_of_one_number_a_row(rows, N, K, ranges):
    """A weight read out by one-hot tokens is what it was."""
    assert _in_two_pieces(rows, N, K) == ranges
    w, at = _rand(N, K, seed=6).cuda(), torch.randint(0, K, (rows,), generator=torch.Generator().manual_seed(9)).cuda()
    x = torch.zeros(rows, K, device="cuda")
    x[torch.arange(rows, device="cuda"), at] = 1.0
    assert torch.equal(M.row_gemm(x, w), w[:, at].T)


@pytest.mark.parametrize("rows,dtype", [(24, torch.bfloat16), (192, torch.float32)])
def test_products_that_the_kernel_does_not_take(rows, dtype):
    """A row repeated, rows that overlap, one or no output, no channel, autocast: as torch.mm has them."""
    K = 64
    base, w = _rand(rows * 8 + K, seed=1).to(dtype).cuda(), _rand(40, K, seed=2).to(dtype).cuda()
    forms = [(base[:K].expand(rows, K), w), (base.as_strided((rows, K), (8, 1)), w), (base[:rows * 8].view(rows, 8).repeat(1, 8), base[:K].expand(3, K)),
             (base[:rows * 8].view(rows, 8), base.as_strided((1, 8), (0, 1))), (base[:rows * 8].view(rows, 8), w[:0, :8]),
             (base[:rows * 8].view(rows, 8)[:, :0], w[:, :0])]
    for x, y in forms:
        assert torch.equal(M.product(x, y), torch.mm(x, y.t()))
    with torch.autocast("cuda", dtype=torch.float16):
        assert M.product(base[:rows * 8].view(rows, 8), w[:, :8]).dtype == torch.float16
    with pytest.raises(RuntimeError):
        M.row_gemm(base[:rows * 8].view(rows, 8), w[:, :8].cpu())
