"""Attention of several tokens in the plain decoder: one call against plain torch in 64 bits, and the model against the path
that torch operations take."""
import pytest
import torch

from decdec_amd import decode_ops as D, generate as G
from decdec_amd.model import apply_rope, rope_tables

pytestmark = pytest.mark.gpu


def _reference(q, k, v, pos):
    """q [H, S, D] on cache rows 0 .. pos[i] of k, v [G, max_seq, D]."""
    H, G = q.shape[0], k.shape[0]
    k, v = k.double().repeat_interleave(H // G, 0), v.double().repeat_interleave(H // G, 0)
    s = torch.stack([q[h].double() @ k[h].T.contiguous() for h in range(H)]) / q.shape[-1] ** 0.5
    s = s.masked_fill(torch.arange(k.shape[1], device=q.device)[None, None] > pos[None, :, None], -float("inf"))
    return torch.stack([torch.softmax(s[h], -1) @ v[h] for h in range(H)]).transpose(0, 1).reshape(pos.numel(), -1)


# rows at the edges of 16-, 64- and 128-query blocks, key counts at the edges of 64-key tiles, a past, positions out of order
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,Hkv,hd,max_seq,start,S,shuffle", [
    (8, 2, 64, 256, 0, 2, False), (8, 2, 64, 200, 61, 17, False), (4, 4, 128, 129, 0, 129, False), (32, 8, 128, 1100, 0, 1027, False),
    (40, 10, 128, 640, 63, 65, False), (32, 8, 128, 2048, 1500, 64, False), (5, 1, 64, 320, 0, 300, True), (64, 8, 128, 600, 7, 513, True)])
def test_prompt_attention(H, Hkv, hd, max_seq, start, S, shuffle, dt):
    g = torch.Generator(device="cuda").manual_seed(S)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")
    cos, sin = (t.to(dt) for t in rope_tables(hd, max_seq, 10000.0, "cuda"))
    kc, vc = rand(1, Hkv, max_seq, hd).to(dt), rand(1, Hkv, max_seq, hd).to(dt)
    k0, v0 = kc.clone(), vc.clone()
    pos = start + torch.arange(S, device="cuda")
    if shuffle:
        pos = pos[torch.randperm(S, generator=g, device="cuda")]
    qkv = (rand(S, (H + 2 * Hkv) * hd) * 1.5).to(dt)
    kt, vt = kc.clone(), vc.clone()
    out = D.prompt_attention(qkv, cos[pos], sin[pos], pos, kc, vc, H, Hkv)
    assert torch.equal(D.prompt_attention(qkv, cos, sin, pos, kt, vt, H, Hkv, tables=True), out) and torch.equal(kt, kc) and torch.equal(vt, vc)
    heads = qkv.view(S, H + 2 * Hkv, hd).transpose(0, 1)
    turned = apply_rope(heads[:H + Hkv].double(), cos[pos].double(), sin[pos].double())
    unit = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    # two products and a sum in fp32, rounded once
    assert ((kc[0, :, pos].double() - turned[H:]).abs() <= unit * turned[H:].abs() + 2.0 ** -21 * qkv.abs().max().double()).all()
    assert torch.equal(vc[0, :, pos], heads[H + Hkv:])
    keep = torch.ones(max_seq, dtype=torch.bool, device="cuda")
    keep[pos] = False
    assert torch.equal(kc[:, :, keep], k0[:, :, keep]) and torch.equal(vc[:, :, keep], v0[:, :, keep])
    want = _reference(turned[:H].to(dt), kc[0], vc[0], pos)
    # an output is rounded once; a query element that the kernel's fp32 rotation rounds the other way moves a score by a unit
    assert float((out.double() - want).abs().max()) <= 2 * unit * float(vc.abs().max())


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128])
def test_a_position_that_the_cache_does_not_have_is_seen_in_its_row_alone(hd, dt):
    H, Hkv, max_seq, S = 4, 2, 96, 20
    g = torch.Generator(device="cuda").manual_seed(hd)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda").to(dt)
    cos, sin = (t.to(dt) for t in rope_tables(hd, max_seq, 10000.0, "cuda"))
    qkv, kc, vc = rand(S, (H + 2 * Hkv) * hd), rand(1, Hkv, max_seq, hd), rand(1, Hkv, max_seq, hd)
    pos = 60 + torch.arange(S, device="cuda")
    bad = torch.zeros(S, dtype=torch.bool, device="cuda")
    for row, at in ((3, -1), (9, max_seq), (16, 2 ** 32 + 5), (17, -2 ** 63)):
        pos[row], bad[row] = at, True
    kw, vw = kc.clone(), vc.clone()
    want = D.prompt_attention(qkv[~bad], cos, sin, pos[~bad], kw, vw, H, Hkv, tables=True)
    out = D.prompt_attention(qkv, cos, sin, pos, kc, vc, H, Hkv, tables=True)
    assert out[bad].isnan().all() and torch.equal(kc, kw) and torch.equal(vc, vw)
    # other rows beside them in a wave: both are within two units of the 64-bit result, as above
    assert float((out[~bad].double() - want.double()).abs().max()) <= 4 * (2.0 ** -11 if dt == torch.float16 else 2.0 ** -8) * float(vc.abs().max())


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [14, 22, 26])
def test_many_small_weights_keep_their_part(bits, dt):
    """One key far ahead of 3000 others, each of which weighs about 2 ** -bits of it and all of whose values are larger."""
    H, Hkv, hd, S = 4, 2, 128, 3000
    g = torch.Generator(device="cuda").manual_seed(bits)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")
    qkv = torch.cat((torch.ones(S, H, hd, device="cuda"), 0.01 * rand(S, Hkv, hd), rand(S, Hkv, hd).abs() + 1), 1)
    qkv[0, H:H + Hkv], qkv[0, H + Hkv:] = bits * 0.6931 / hd ** 0.5, 1e-3
    qkv = qkv.to(dt)
    cos, sin = torch.ones(S, hd, device="cuda", dtype=dt), torch.zeros(S, hd, device="cuda", dtype=dt)
    kc, vc = (torch.zeros(1, Hkv, S, hd, device="cuda", dtype=dt) for _ in range(2))
    pos = torch.arange(S, device="cuda")
    out = D.prompt_attention(qkv.view(S, -1), cos, sin, pos, kc, vc, H, Hkv)
    want = _reference(qkv[:, :H].transpose(0, 1), kc[0], vc[0], pos)
    # one rounding of the output.  A weight of 2 ** -26 keeps 2 ** -13 of itself in fp16 (the trailing part ends at 2 ** -24 of a
    # scale of 2 ** 15; in bf16 three parts are the 32-bit number), and all values have one sign; scores are exact to 2 ** -18
    unit = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    assert ((out.double() - want).abs() <= (unit + 2.0 ** -12) * want.abs()).all()


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_keys_that_a_query_may_not_see_do_not_matter(bad, dt):
    """Later tokens of the prompt, and what the cache holds behind it: in the tiles of the queries and past them."""
    H, Hkv, hd, S, max_seq, start = 8, 2, 64, 150, 420, 70
    g = torch.Generator(device="cuda").manual_seed(1)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda").to(dt)
    cos, sin = (t.to(dt)[start:start + S] for t in rope_tables(hd, max_seq, 10000.0, "cuda"))
    qkv, pos, k0, v0 = rand(S, H + 2 * Hkv, hd), start + torch.arange(S, device="cuda"), rand(1, Hkv, max_seq, hd), rand(1, Hkv, max_seq, hd)
    run = lambda x, k: D.prompt_attention(x.view(S, -1), cos, sin, pos, k, v0.clone(), H, Hkv)
    clean = run(qkv, k0.clone())
    behind = k0.clone()
    behind[:, :, start:] = bad
    assert torch.equal(run(qkv, behind), clean) and torch.isfinite(clean).all()
    for t in (1, 58, 59, 100, 149):                        # the first token whose key is bad
        later = qkv.clone()
        later[t:, H:H + Hkv] = bad
        assert torch.equal(run(later, behind.clone())[:t], clean[:t])


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_keys_infinitely_far_below_all_others(dt):
    """Scores of minus infinity weigh nothing, also where a tile has no other ones."""
    H, Hkv, hd, S, start = 4, 2, 128, 90, 70
    g = torch.Generator(device="cuda").manual_seed(2)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda").to(dt)
    qkv = rand(S, H + 2 * Hkv, hd)
    qkv[:, :H] = qkv[:, :H].abs() + 0.01
    cos, sin = torch.ones(S, hd, device="cuda", dtype=dt), torch.zeros(S, hd, device="cuda", dtype=dt)
    kc, vc, pos = rand(1, Hkv, start + S, hd), rand(1, Hkv, start + S, hd), start + torch.arange(S, device="cuda")
    kc[:, :, :start] = -float("inf")
    out = D.prompt_attention(qkv.view(S, -1), cos, sin, pos, kc, vc, H, Hkv)
    want = _reference(qkv[:, :H].transpose(0, 1), kc[0], vc[0], pos)
    unit = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    assert float((out.double() - want).abs().max()) <= 2 * unit * float(vc.abs().max())


@pytest.mark.parametrize("fmt,bits,dt", [("sqllm", 4, torch.float16), ("anyprec", 3, torch.bfloat16), ("lutgemm", 3, torch.float16), ("sqllm", 3, torch.bfloat16)])
@pytest.mark.parametrize("cut", [[40], [1, 39], [13, 2, 25]])
def test_prompt_through_kernels_is_the_prompt_through_torch(cut, fmt, bits, dt, monkeypatch):
    """Portions of a prompt, logits and caches, against the torch operations (which autograd mode still takes)."""
    m = G.build_model("tiny-llama-test", fmt, bits, dtype=dt)
    tokens = torch.randint(0, m.config.vocab_size, (40,), generator=torch.Generator().manual_seed(0)).cuda()
    m.setup_caches(1, 72)
    calls, plain = [], D.prompt_attention
    monkeypatch.setattr(D, "prompt_attention", lambda *a: calls.append(a[0].shape[0]) or plain(*a))
    with torch.enable_grad():
        want = m(tokens[None], torch.arange(40, device="cuda"))[0, -1].detach()
    assert not calls
    kept = []
    with torch.no_grad():
        for b in m.layers:
            for c in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache):
                kept.append((c, c.clone()))
                c.fill_(0.75)                              # what the second pass does not write is not the first one's
    s = G.Session(m, 72)
    at = 0
    for n in cut:
        got = s.feed(tokens[at:at + n], [n - 1])[0]
        at += n
    assert calls == [n for n in cut if n > 1 for _ in m.layers]
    # sublayers round their activations a few times, in places that differ: some units of the storage type
    unit = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    off = lambda a, b: float((a.detach().float() - b.detach().float()).norm() / b.detach().float().norm())
    assert off(got, want) < max(1e-2, 8 * unit)
    for c, was in kept:
        assert off(c[:, :, :40], was[:, :, :40]) < max(5e-3, 4 * unit) and (c[:, :, 40:] == 0.75).all()
