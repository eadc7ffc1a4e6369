"""Prompts through the quantised layers and the plain decoder: which calls take the library's kernels, and that those which do not
come out as torch operations on the dense weight give them."""
import pytest
import torch

from decdec_amd import decode_ops, ext, formats as F, generate as G
from decdec_amd.linear import APLinear, LUTGEMMLinear, SQLLMLinear
from decdec_amd.model import TransformerBlock

pytestmark = pytest.mark.gpu


def _words(*shape):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int64).to(torch.int32).cuda()


def _layer(fmt, K, N, bits, dtype, group=128):
    """(layer, its dense weight by torch operations)."""
    if fmt == "lutgemm":
        l = LUTGEMMLinear(K, N, bits, group, dtype=dtype)
        l.qweight.copy_(_words(*l.qweight.shape))
        l.alpha.copy_(torch.rand(l.alpha.shape) * 0.1)
        l.q_bias.copy_(torch.randn(l.q_bias.shape) * 0.1)
        return l, F.dequant_bcq(l.qweight, l.alpha, l.q_bias, group).to(dtype)
    l = (APLinear if fmt == "anyprec" else SQLLMLinear)(K, N, bits, dtype=dtype)
    l.qweight.copy_(_words(*l.qweight.shape))
    l.lut.copy_(torch.randn(l.lut.shape))
    return l, F.dequant_lut(F.unpack_anyprec(l.qweight, bits), l.lut) if fmt == "anyprec" else F.dequant_sqllm(l.qweight, l.lut, bits)


def _close(got, x, w):
    """A product of 16-bit numbers, summed in 32 bits and rounded once, against 64 bits."""
    want, size = x.double() @ w.double().T.contiguous(), x.double().abs() @ w.double().abs().T.contiguous()
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}.get(got.dtype, 2.0 ** -24)
    assert got.shape == want.shape and ((got.double() - want).abs() <= unit * want.abs() + 2.0 ** -19 * size + 1e-30).all()


@pytest.mark.parametrize("tokens", [20, 300])
@pytest.mark.parametrize("fmt", ["lutgemm", "sqllm"])
def test_traced_prompt(fmt, tokens):
    """A trace replays the products of its inputs, and new ones."""
    torch.manual_seed(tokens)
    layer, w = _layer(fmt, 256, 72, 3, torch.float16)
    a, b = (torch.randn(1, tokens, 256, device="cuda", dtype=torch.float16) for _ in range(2))
    with torch.no_grad():
        traced = torch.jit.trace(lambda x: layer.gemm(x), a, check_trace=False)
        for x in (a, b):
            _close(traced(x), x, w)


def test_products_refuse_tables_elsewhere():
    """An address of the host is never handed to a kernel."""
    x = torch.zeros(4, 128, device="cuda", dtype=torch.float16)
    tables = torch.zeros(16, 16, device="cuda", dtype=torch.float16)
    alpha, bias = torch.zeros(1, 4, 16, device="cuda", dtype=torch.float16), torch.zeros(1, 16, device="cuda", dtype=torch.float16)
    calls = [(ext.sqllm_gemm, [_words(16, 16), tables, 4]), (ext.anyprec_gemm, [_words(4, 16, 4), tables, 4]),
             (ext.lutgemm_gemm, [_words(4, 4, 16), alpha, bias, 4, 128])]
    for op, args in calls:
        op(x, *args)
        for i, t in enumerate(args):
            if torch.is_tensor(t):
                with pytest.raises(RuntimeError):
                    op(x, *args[:i], t.cpu(), *args[i + 1:])
        with pytest.raises(RuntimeError):
            op(x.cpu(), *args)


@pytest.mark.parametrize("tokens", [2, 300])
@pytest.mark.parametrize("K", [8, 40, 4104])
def test_prompt_of_a_squeezellm_layer_without_whole_units(K, tokens):
    """4 bits hold any multiple of eight channels; the kernels take units of 32."""
    torch.manual_seed(K)
    layer, w = _layer("sqllm", K, 24, 4, torch.float16)
    x = torch.randn(1, tokens, K, device="cuda", dtype=torch.float16)
    _close(layer(x), x, w)


@pytest.mark.parametrize("tokens", [2, 300])
@pytest.mark.parametrize("fmt", ["lutgemm", "sqllm"])
def test_prompt_in_64_bits(fmt, tokens):
    """A type that the kernels do not have goes through torch operations."""
    torch.manual_seed(tokens)
    layer, w = _layer(fmt, 256, 24, 4, torch.float64)
    x = torch.randn(1, tokens, 256, device="cuda", dtype=torch.float64)
    got = layer(x)
    assert got.dtype == torch.float64
    _close(got, x, w)


@pytest.mark.parametrize("fmt", ["anyprec", "lutgemm", "sqllm"])
def test_product_of_no_tokens(fmt):
    layer, _ = _layer(fmt, 256, 24, 4, torch.float16)
    x = torch.zeros(1, 0, 256, device="cuda", dtype=torch.float16)
    assert layer.gemm(x).shape == (1, 0, 24)
    if fmt == "lutgemm":                                   # nor of no outputs
        none, _ = _layer(fmt, 256, 0, 4, torch.float16)
        for tokens in (3, 300):
            assert none.gemm(torch.zeros(1, tokens, 256, device="cuda", dtype=torch.float16)).shape == (1, tokens, 0)


@pytest.mark.parametrize("tokens", [20, 300])
@pytest.mark.parametrize("fmt", ["anyprec", "lutgemm", "sqllm"])
def test_autocast_chooses_the_type_of_a_product(fmt, tokens):
    torch.manual_seed(tokens)
    layer, w = _layer(fmt, 256, 72, 3, torch.float16)
    x = torch.randn(1, tokens, 256, device="cuda", dtype=torch.float16)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        got = layer(x)
        assert got.dtype == torch.bfloat16
    _close(got, x.to(torch.bfloat16), w.to(torch.bfloat16))


def test_autocast_keeps_a_prompt_on_torch_operations():
    m = G.build_model("tiny-llama-test", "sqllm", 4)
    m.setup_caches(1, 72)
    x, pos = torch.zeros(1, 20, m.config.dim, device="cuda", dtype=torch.float16), torch.arange(20, device="cuda")
    with torch.no_grad():
        assert m._prompt_on_kernels(x, pos)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not m._prompt_on_kernels(x, pos)


def test_hooks_see_every_module_of_a_prompt():
    """Norms and the head run inside kernels, unless a hook, of theirs or on all modules, wants to see them."""
    m = G.build_model("tiny-llama-test", "sqllm", 4)
    m.setup_caches(1, 72)
    tokens = torch.zeros(1, 20, dtype=torch.int64, device="cuda")
    run = lambda: m(tokens, torch.arange(20, device="cuda"), want=[19])
    n = len(m.layers)
    with torch.no_grad():
        plain, seen = run(), []
        handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, args, out: seen.append(type(mod).__name__))
        try:
            hooked = run()
        finally:
            handle.remove()
        assert seen.count("RMSNorm") == 2 * n + 1 and seen.count("Linear") == 1
        own = []
        handles = [x.register_forward_hook(lambda mod, args, out: own.append(mod)) for x in (m.layers[0].post_attention_layernorm, m.output)]
        run()
        assert own == [m.layers[0].post_attention_layernorm, m.output]
        for h in handles:
            h.remove()
    assert float((plain - hooked).float().norm() / plain.float().norm()) < 1e-2


@pytest.fixture
def steps(monkeypatch):
    """The blocks that a prompt passed through from block to block."""
    seen, step = [], TransformerBlock.prompt_step
    monkeypatch.setattr(TransformerBlock, "prompt_step", lambda self, *args: seen.append(self) or step(self, *args))
    return seen


def _by_torch_operations(m, *args, **kwargs):
    kernels, m.decode_kernels = m.decode_kernels, False
    try:
        return m(*args, **kwargs)
    finally:
        m.decode_kernels = kernels


def test_prompt_with_sums_and_norms_in_one_pass(steps):
    """The same logits and caches as with blocks that are called (a hook on one of them sees to it), for all places and for some; a norm
    or a block of a user's own is called."""
    m = G.build_model("tiny-llama-test", "sqllm", 4)
    tokens, pos = torch.randint(0, m.config.vocab_size, (1, 37), device="cuda"), torch.arange(37, device="cuda")
    blocks = list(m.layers)
    with torch.no_grad():
        for want in (None, [36], [3, 4, 5], [1, 9]):
            m.setup_caches(1, 72)
            steps.clear()
            got, keys = m(tokens, pos, want=want), [b.attention.kv_cache.k_cache.clone() for b in m.layers]
            assert steps == ([] if want == [1, 9] else blocks)                  # places that do not follow each other: blocks are called
            seen = []
            steps.clear()
            handle = m.layers[-1].register_forward_hook(lambda mod, args, out: seen.append(mod))
            ref = m(tokens, pos, want=want)
            handle.remove()
            assert seen == [m.layers[-1]] and steps == [] and got.shape == ref.shape
            assert float((got - ref).float().norm() / ref.float().norm()) < 5e-3
            assert all(float((a - b.attention.kv_cache.k_cache).float().norm() / a.float().norm()) < 5e-3 for a, b in zip(keys, m.layers))
            ref = _by_torch_operations(m, tokens, pos, want=want)
            assert float((got - ref).float().norm() / ref.float().norm()) < 5e-3
        calls = []
        norm = m.layers[0].input_layernorm
        norm.forward = lambda x, f=norm.forward: calls.append(x.shape) or f(x)
        m(tokens, pos, want=[36])
        assert calls == [(1, 37, m.config.dim)] and steps == []


def test_prompt_of_blocks_whose_parts_were_changed(steps):
    """A hook that changes a projection's result, and rotary tables longer than the caches: what the blocks' own calls give."""
    m = G.build_model("tiny-llama-test", "sqllm", 4)
    m.setup_caches(1, 72)
    tokens, pos = torch.randint(0, m.config.vocab_size, (1, 37), device="cuda"), torch.arange(37, device="cuda")
    with torch.no_grad():
        plain, cos, sin = m(tokens, pos), m.rope_cos, m.rope_sin
        assert steps == list(m.layers)
        steps.clear()
        m.rope_cos, m.rope_sin = torch.cat((cos, cos)), torch.cat((sin, sin))
        assert float((m(tokens, pos) - plain).float().norm() / plain.float().norm()) < 5e-3
        m.rope_cos, m.rope_sin = cos, sin
        handle = m.layers[-1].feed_forward.w2.register_forward_hook(lambda mod, args, out: out[:, :1])      # added to every row
        changed, ref = m(tokens, pos), _by_torch_operations(m, tokens, pos)
        handle.remove()
    assert changed.shape == plain.shape and not torch.equal(changed, plain) and steps == []
    assert float((changed - ref).float().norm() / ref.float().norm()) < 5e-3


def test_prompt_of_a_projection_class_of_a_user(steps):
    """Results that start between two pieces of 8 bytes, and one row for all: added as torch adds them."""
    class Apart(SQLLMLinear):
        def forward(self, x, **kwargs):
            y = super().forward(x, **kwargs)
            room = torch.empty(y.numel() + 1, dtype=y.dtype, device=y.device)
            return room[1:].view(y.shape).copy_(y)

    class OneRow(SQLLMLinear):
        def forward(self, x, **kwargs):
            return super().forward(x, **kwargs)[:, :1]
    m = G.build_model("tiny-llama-test", "sqllm", 4)
    m.setup_caches(1, 72)
    tokens, pos = torch.randint(0, m.config.vocab_size, (1, 37), device="cuda"), torch.arange(37, device="cuda")
    with torch.no_grad():
        for kind in (SQLLMLinear, Apart, OneRow):
            for b in m.layers:
                b.feed_forward.w2.__class__ = kind
            for want in (None, [36], [3, 4, 5], [1, 9]):
                steps.clear()
                got = m(tokens, pos, want=want)
                assert steps == ([] if want == [1, 9] else list(m.layers))
                ref = _by_torch_operations(m, tokens, pos, want=want)
                assert got.shape == ref.shape and float((got - ref).float().norm() / ref.float().norm()) < 5e-3, (kind, want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt,bits", [("anyprec", 3), ("anyprec", 4), ("anyprec", 6), ("lutgemm", 3), ("lutgemm", 4), ("lutgemm", 2), ("sqllm", 3), ("sqllm", 4)])
def test_which_prompt_takes_which_kernel(fmt, bits, dtype, monkeypatch):
    """Up to 256 tokens on the packed weight, more on its expansion; what these kernels do not take, on torch operations."""
    torch.manual_seed(bits)
    layer, w = _layer(fmt, 256, 72, bits, dtype)
    taken = []
    for name in (f"{fmt}_gemm", f"{fmt}_dequant"):
        op = getattr(ext, name)
        monkeypatch.setattr(ext, name, lambda *a, op=op, name=name: taken.append(name.split("_")[1]) or op(*a))

    def route(x, *expected):
        taken.clear()
        with torch.no_grad():
            _close(layer(x), x, w)
        assert tuple(taken) == expected, (taken, expected)
    x = torch.randn(1, 257, 256, device="cuda").to(dtype)
    packed = ("gemm",) if bits in (3, 4) else ("dequant",)
    for tokens in (2, 77, 256):
        route(x[:, :tokens].contiguous(), *packed)
    route(x, "dequant")
    apart = torch.empty(20 * 256 + 1, device="cuda", dtype=dtype)[1:].view(1, 20, 256)             # starts between two pieces of 16 bytes
    route(apart.copy_(x[:, :20]), "dequant")
    route(x[:, :40:2], "dequant")                                                                  # rows apart
    layer.qweight = layer.qweight.as_subclass(type("Words", (torch.Tensor,), {}))
    if fmt != "anyprec":                                                                           # whose expansion always was this kernel
        route(x[:, :20].contiguous())
        route(x)


@pytest.mark.parametrize("tokens", [2, 37, 256, 257])
@pytest.mark.parametrize("fmt,bits,dtype", [("anyprec", 3, torch.bfloat16), ("anyprec", 4, torch.float16), ("anyprec", 6, torch.float16), ("lutgemm", 3, torch.float16),
                                            ("lutgemm", 4, torch.bfloat16), ("sqllm", 3, torch.bfloat16), ("sqllm", 4, torch.float16)])
def test_prompt_of_blocks_in_a_call_each(fmt, bits, dtype, tokens, monkeypatch):
    """The linear parts of a block in one call ahead of the attention and one behind it: the bits that the layers' own calls give (a hook on one sees to
    it), for the prompts whose products are all packed."""
    m = G.build_model("tiny-llama-test", fmt, bits, dtype=dtype)
    ids, pos = torch.randint(0, m.config.vocab_size, (1, tokens), device="cuda"), torch.arange(tokens, device="cuda")
    parts, back = [], decode_ops.prompt_back
    monkeypatch.setattr(decode_ops, "prompt_back", lambda *args: parts.append(args) or back(*args))
    m.setup_caches(1, 264)
    with torch.no_grad():
        got, kept = m(ids, pos), [(b.attention.kv_cache.k_cache.clone(), b.attention.kv_cache.v_cache.clone()) for b in m.layers]
        assert len(parts) == (len(m.layers) if bits in (3, 4) and tokens <= 256 else 0)
        parts.clear()
        handles = [b.attention.wqkv.register_forward_hook(lambda mod, args, out: None) for b in m.layers]
        want = m(ids, pos)
        assert not parts and torch.equal(got, want)
        for b, (k, v) in zip(m.layers, kept):
            assert torch.equal(b.attention.kv_cache.k_cache, k) and torch.equal(b.attention.kv_cache.v_cache, v)
        for h in handles:
            h.remove()


@pytest.mark.parametrize("arena", [True, False])
@pytest.mark.parametrize("fmt,dtype", [("sqllm", torch.float16), ("lutgemm", torch.bfloat16)])
def test_steps_that_begin_in_one_launch(fmt, dtype, arena, monkeypatch):
    """Embedding, first norm and the arena's zeros by one kernel: the bits of the calls by themselves, which are made where somebody sees the embedding,
    where it is another module, or where a gradient is asked for.  (The products add up in any order: 16 roundings of the type for two blocks' logits.)"""
    m = G.build_model("tiny-llama-test", fmt, 4, dtype=dtype)
    if not arena:
        m.output_arena = None
        for layer in m.layers:
            for l in layer.dec_linears():
                l.external_zero = False
    m.setup_caches(1, 16)
    opened, op = [], decode_ops.open_step
    monkeypatch.setattr(decode_ops, "open_step", lambda *args: op(*args) or opened.append((args[4].clone(), args[5].clone())))
    idx = torch.randint(0, m.config.vocab_size, (4, 1, 1), device="cuda")

    def steps():
        opened.clear()
        return torch.cat([m(t, torch.tensor([i], device="cuda")) for i, t in enumerate(idx)])

    def close(x):
        return bool((x.float() - want.float()).abs().max() <= 16 * torch.finfo(dtype).eps * want.float().abs().max())
    with torch.no_grad():
        got = steps()
        assert len(opened) == len(idx)
        for t, (h, n) in zip(idx, opened):
            norm, first, want = m.layers[0].input_layernorm, m.tok_embeddings(t), torch.empty_like(h)
            decode_ops.add_rmsnorm(first, None, norm.weight, None, want, norm.eps)
            assert torch.equal(h, first) and torch.equal(n, want)
        handle = m.tok_embeddings.register_forward_hook(lambda mod, args, out: None)
        want = steps()
        assert not opened and close(got)
        handle.remove()
        kept, m.tok_embeddings = m.tok_embeddings, torch.nn.Sequential(m.tok_embeddings)
        assert close(steps()) and not opened
        m.tok_embeddings = kept
        m(idx[0].to(torch.int32), torch.tensor([0], device="cuda"))
        assert not opened
    kept.weight.requires_grad_(True)
    assert close(steps().detach()) and not opened


@pytest.mark.parametrize("fmt,bits,dtype", [("sqllm", 4, torch.float16), ("sqllm", 3, torch.bfloat16), ("anyprec", 3, torch.float16)])
def test_steps_whose_products_make_their_activations(fmt, bits, dtype, monkeypatch):
    """Norms and gates in the launches of the SqueezeLLM products behind them, from the second block's norm on: the logits of the launches apart (products add up
    in any order: 16 roundings of the type for two blocks' logits), which are made where somebody sees a call, changes one, or asks for compensation."""
    m = G.build_model("tiny-llama-test", fmt, bits, dtype=dtype)
    m.setup_caches(1, 16)
    made = []
    for name in ("norm_product", "gate_product"):
        op = getattr(decode_ops, name)
        monkeypatch.setattr(decode_ops, name, lambda *args, op=op, name=name: made.append(name) or op(*args))
    idx = torch.randint(0, m.config.vocab_size, (4, 1, 1), device="cuda")

    def steps():
        made.clear()
        return torch.cat([m(t, torch.tensor([i], device="cuda")) for i, t in enumerate(idx)])

    def close(x):
        return bool((x.float() - want.float()).abs().max() <= 16 * torch.finfo(dtype).eps * want.float().abs().max())
    L = len(m.layers)
    with torch.no_grad():
        got = steps()
        assert (made.count("norm_product"), made.count("gate_product")) == ((4 * (2 * L - 1), 4 * L) if fmt == "sqllm" else (0, 0))
        keep = [h for b in m.layers for h in (b.attention.register_forward_hook(lambda *a: None), b.feed_forward.register_forward_hook(lambda *a: None))]
        want = steps()
        assert not made and close(got)
        for h in keep:
            h.remove()
        if fmt != "sqllm":
            return
        b = m.layers[-1]
        # one of the two of a feed-forward alone
        b.feed_forward.w1w3.forward = type(b.feed_forward.w1w3).forward.__get__(b.feed_forward.w1w3)
        assert close(steps()) and (made.count("norm_product"), made.count("gate_product")) == (4 * (2 * L - 2), 4 * L)
        del b.feed_forward.w1w3.forward
        handle = b.post_attention_layernorm.register_forward_hook(lambda *a: None)
        assert close(steps()) and (made.count("norm_product"), made.count("gate_product")) == (4 * (2 * L - 2), 4 * L)
        handle.remove()
        b.feed_forward.w2.external_zero, b.feed_forward.w2.output = False, torch.zeros_like(b.feed_forward.w2.output)
        assert close(steps()) and (made.count("norm_product"), made.count("gate_product")) == (4 * (2 * L - 1), 4 * (L - 1))


def test_a_step_behind_a_changed_option(monkeypatch):
    """Fewer ranges of channels, set between two steps of the same layers: a product that has no room for its activations any more takes the launches apart."""
    from decdec_amd import _lib
    from decdec_amd.model import ModelArgs, Transformer
    m = Transformer(torch.float16, ModelArgs(n_layer=1, n_head=2, n_local_heads=1, dim=256, intermediate_size=8192, vocab_size=64), linear_class=SQLLMLinear,
                    linear_kwargs={"bitwidth": 4, "dtype": torch.float16})
    G.init_random_weights(m, 3)
    m.share_output_arena()
    m.eval().setup_caches(1, 16)
    made, op = [], decode_ops.gate_product
    monkeypatch.setattr(decode_ops, "gate_product", lambda *args: made.append(1) or op(*args))
    idx, pos = torch.tensor([[7]], device="cuda"), torch.tensor([0], device="cuda")
    with torch.no_grad():
        want = m(idx, pos)
        assert len(made) == 1
        _lib.set_option("gemv_max_k_ranges", 1)
        try:
            got = m(idx, pos)
            assert len(made) == 1
        finally:
            _lib.set_option("gemv_max_k_ranges", 0)
        again = m(idx, pos)
        assert len(made) == 2
    for x in (got, again):                                 # products add up in any order: 16 roundings of the type
        assert (x.float() - want.float()).abs().max() <= 16 * torch.finfo(torch.float16).eps * want.float().abs().max()
