"""Which calls may hand tensors to the library by address: the conditions, on the CPU."""
import pytest
import torch
from torch.utils.flop_counter import FlopCounterMode

from decdec_amd import ext


def test_tracing_sees_torch_operations():
    """A trace that passed a kernel by would replay memory that nothing wrote."""
    seen = []

    def f(x):
        seen.append(ext.watched())
        return x + 1
    torch.jit.trace(f, torch.zeros(2), check_trace=False)
    assert seen and all(seen) and not ext.watched()


def test_vmap_modes_and_forward_mode_see_torch_operations():
    seen = []

    def f(x):
        seen.append(ext.watched())
        return x * 2
    torch.func.vmap(f)(torch.zeros(3, 2))
    torch.func.jvp(f, (torch.zeros(2),), (torch.ones(2),))
    with torch.autograd.forward_ad.dual_level():
        f(torch.zeros(2))
    with FlopCounterMode(display=False):
        f(torch.zeros(2))
    assert len(seen) == 4 and all(seen) and not ext.watched()


def test_plain_tensors():
    cpu, w = -1, torch.zeros(4, 6)

    class Wrapped(torch.Tensor):
        pass
    assert ext.plain(cpu, w, torch.nn.Parameter(w, requires_grad=False))
    assert not ext.plain(cpu, w.t()) and not ext.plain(cpu, w, w.as_subclass(Wrapped)) and not ext.plain(0, w)
    leaf = w.clone().requires_grad_()
    assert not ext.plain(cpu, leaf)
    with torch.no_grad():
        assert ext.plain(cpu, leaf)
    assert not ext.on_kernels(w.device, w)


def test_a_default_device_is_no_watcher():
    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with torch.device("cpu"):
        assert not ext.watched()
        with Mode():
            assert ext.watched()
    with Mode(), torch.device("cpu"):
        assert ext.watched()
    torch.set_default_device("cpu")
    try:
        assert not ext.watched()
    finally:
        torch.set_default_device(None)


class Elsewhere(torch.Tensor):
    """As a tensor of GPU 1 answers."""

    def get_device(self):
        return 1


def test_rotary_tables_left_on_another_gpu_are_not_read_by_address():
    """Caches are buffers and move with a model, the tables are attributes and stay."""
    from decdec_amd.model import _read_at_positions, rope_tables
    x, (cos, sin) = torch.zeros(1, 5, 64), rope_tables(64, 16, 10000.0)
    with torch.no_grad():
        assert _read_at_positions(x, cos, sin)
        assert not _read_at_positions(x, cos.as_subclass(Elsewhere), sin) and not _read_at_positions(x, cos, sin.as_subclass(Elsewhere))
        assert not _read_at_positions(x, cos, sin[:8]) and not _read_at_positions(x, cos.t().contiguous().t(), sin)


def test_blocks_that_somebody_watches_are_called():
    from decdec_amd.cache import KVCache
    from decdec_amd.model import ModelArgs, TransformerBlock

    class Layer(torch.nn.Module):
        def __init__(self, in_features, out_features, bias):
            super().__init__()
            self.out_features, self.dtype = out_features, torch.float32
    config = ModelArgs.from_name("tiny-llama-test")
    block, x = TransformerBlock(config, Layer, {}), torch.zeros(1, 5, config.dim)
    block.attention.kv_cache = KVCache(1, 16, config.n_local_heads, config.head_dim, x.dtype, x.device)
    assert block.steps_over(x, 16) and not block.steps_over(x, 24)
    for part in (block, block.attention, block.feed_forward, block.attention.wo, block.feed_forward.w2, block.input_layernorm):
        for watch in (part.register_forward_hook, part.register_forward_pre_hook, torch.nn.modules.module.register_module_forward_hook):
            handle = watch(lambda *args: None)
            assert not block.steps_over(x, 16)
            handle.remove()
        part.forward = lambda *args: None
        assert not block.steps_over(x, 16)
        del part.forward
        assert block.steps_over(x, 16)


def test_tensors_of_two_gpus_are_refused():
    from decdec_amd import decode_ops

    class Here(Elsewhere):
        is_cuda = True

        def get_device(self):
            return 0
    half = lambda *s: torch.zeros(*s, dtype=torch.float16)
    here, there = (lambda t: t.as_subclass(Here)), (lambda t: t.as_subclass(type("There", (Here,), {"get_device": lambda self: 1})))
    args = [half(3, 3 * 64), half(16, 64), half(16, 64), torch.zeros(3, dtype=torch.int64), half(1, 1, 16, 64), half(1, 1, 16, 64)]
    for i in range(6):
        with pytest.raises(RuntimeError, match="of one GPU|on the device"):
            decode_ops.prompt_attention(*[there(t) if i == k else here(t) for k, t in enumerate(args)], 1, 1, tables=True)
    with pytest.raises(RuntimeError, match="of one GPU"):
        decode_ops.prompt_attention(*args, 1, 1, tables=True)


def test_what_a_kernel_writes_counts_as_an_operation_in_place():
    """The version that autograd compares, also in inference mode; what `zero_` refuses, and what it cuts off."""
    out = torch.zeros(1, 1, 4)
    for mode in (torch.enable_grad, torch.no_grad, torch.inference_mode):
        with mode():
            before = out._version
            ext.written(out)
            assert out._version == before + 1
    p = torch.ones(4, requires_grad=True)
    loss = (out * p).sum()
    ext.written(out)
    with pytest.raises(RuntimeError, match="inplace operation"):
        loss.backward()
    with pytest.raises(RuntimeError, match="leaf Variable"):
        ext.written(torch.zeros(2, requires_grad=True))
    with torch.inference_mode():
        made = torch.zeros(2)
        ext.written(made)
    with pytest.raises(RuntimeError, match="inference tensor"):
        ext.written(made)
    out += p                                               # a bias that is learnt
    ext.written(out)
    out += p
    out.sum().backward()
    assert torch.equal(p.grad, torch.ones(4))


def test_layers_that_a_part_of_a_prompt_takes():
    """decdec_packed_layer's numbers of a layer as it is; of what changes its calls or its tensors, none."""
    from decdec_amd.linear import APLinear, LUTGEMMLinear, SQLLMLinear, packed_layer
    at, half = -1, torch.float16

    def make(kind, bits, K=256, N=72, dtype=half, **kw):
        l = kind(K, N, bits, *([128] if kind is LUTGEMMLinear else []), dtype=dtype, device="cpu", **kw)
        table = "alpha" if kind is LUTGEMMLinear else "lut"
        room = torch.zeros(l._buffers[table].numel() + 64, dtype=dtype)      # on the CPU a tensor may start anywhere
        first = (-room.data_ptr() % 16) // room.element_size()
        l._buffers[table] = room[first:first + l._buffers[table].numel()].view(l._buffers[table].shape)
        return l
    for number, kind in enumerate((APLinear, LUTGEMMLinear, SQLLMLinear)):
        for bits in (3, 4):
            l = make(kind, bits)
            table = l._buffers["alpha" if kind is LUTGEMMLinear else "lut"]
            bias = l.q_bias.data_ptr() if kind is LUTGEMMLinear else 0
            expected = (number, bits, 128 if kind is LUTGEMMLinear else 0, 256, 72, l.qweight.data_ptr(), table.data_ptr(), bias)
            with torch.no_grad():
                assert packed_layer(l, 2, half, at) == packed_layer(l, 256, half, at) == expected
                assert packed_layer(l, 257, half, at) is None and packed_layer(l, 2, torch.bfloat16, at) is None and packed_layer(l, 2, half, 0) is None
                for watch in (l.register_forward_hook, l.register_forward_pre_hook):
                    handle = watch(lambda *args: None)
                    assert packed_layer(l, 2, half, at) is None
                    handle.remove()
                for name in ("forward", "gemm"):
                    setattr(l, name, lambda *args: None)
                    assert packed_layer(l, 2, half, at) is None
                    delattr(l, name)
                assert packed_layer(l, 2, half, at) == expected
                words, name = l.qweight, "alpha" if kind is LUTGEMMLinear else "lut"
                l.qweight = words.as_subclass(type("Words", (torch.Tensor,), {}))
                assert packed_layer(l, 2, half, at) is None
                l.qweight = words[..., :-1]
                assert packed_layer(l, 2, half, at) is None
                l.qweight = words.clone().to(torch.int64)
                assert packed_layer(l, 2, half, at) is None
                l.qweight = words
                l._buffers[name] = torch.zeros(table.numel() + 64, dtype=half)[1:1 + table.numel()].view(table.shape)
                assert l._buffers[name].data_ptr() % 16 == 0 or packed_layer(l, 2, half, at) is None
                l._buffers[name] = table
                assert packed_layer(l, 2, half, at) == expected
                assert packed_layer(make(kind, bits, bias=True), 2, half, at) is None
                assert packed_layer(make(type("Own", (kind,), {}), bits), 2, half, at) is None if kind is not LUTGEMMLinear else True
    with torch.no_grad():
        assert packed_layer(make(APLinear, 6), 2, half, at) is None and packed_layer(torch.nn.Linear(8, 8), 2, torch.float32, at) is None
        assert packed_layer(make(SQLLMLinear, 4, K=40), 2, half, at) is None
        wide = make(SQLLMLinear, 4, K=4096, N=4096)
        assert packed_layer(wide, 512, half, at) is not None and packed_layer(wide, 513, half, at) is None
    l = make(SQLLMLinear, 4)
    l._buffers["lut"].requires_grad_()
    assert packed_layer(l, 2, half, at) is None            # its gradient would pass the kernel by


def test_layers_whose_products_make_their_activations():
    """Of one class, seen by nobody, uncompensated, with an output that is cleared elsewhere; by the sizes of the rule."""
    from decdec_amd import decode_ops
    from decdec_amd.linear import APLinear, SQLLMLinear, step_layer
    at, half = -1, torch.float16

    def make(kind=SQLLMLinear, bits=4, K=256, N=72, dtype=half, **kw):
        l = kind(K, N, bits, dtype=dtype, device="cpu", **kw)
        room = torch.zeros(l.lut.numel() + 64, dtype=dtype)                  # on the CPU a tensor may start anywhere
        first = (-room.data_ptr() % 16) // room.element_size()
        l._buffers["lut"] = room[first:first + l.lut.numel()].view(l.lut.shape)
        l.external_zero = True
        return l
    with torch.no_grad():
        for norm in (True, False):
            for bits in (3, 4):
                l = make(bits=bits)
                assert step_layer(l, norm, half, at) and not step_layer(l, norm, torch.bfloat16, at) and not step_layer(l, norm, half, 0)
                for watch in (l.register_forward_hook, l.register_forward_pre_hook):
                    handle = watch(lambda *args: None)
                    assert not step_layer(l, norm, half, at)
                    handle.remove()
                for name, value, old in (("forward", lambda x: x, None), ("external_zero", False, True), ("dec_config", 1, None), ("output", l.output[..., :-1], l.output),
                                         ("qweight", l.qweight[..., :-1], l.qweight), ("lut", l.lut.float(), l.lut)):
                    setattr(l, name, value)
                    assert not step_layer(l, norm, half, at), name
                    delattr(l, name) if name == "forward" else setattr(l, name, old)
                assert step_layer(l, norm, half, at)
            assert not step_layer(make(bias=True), norm, half, at) and not step_layer(make(APLinear), norm, half, at)
            assert not step_layer(make(type("Own", (SQLLMLinear,), {})), norm, half, at) and not step_layer(make(K=40), norm, half, at)
    makes, bf16 = decode_ops.product_makes, torch.bfloat16
    assert makes(True, 4, half, 4096, 28672) and not makes(True, 3, half, 4096, 28672) and not makes(True, 4, bf16, 4096, 28672)
    assert makes(True, 3, bf16, 5120, 7680) and not makes(True, 4, bf16, 5120, 7680) and not makes(True, 4, half, 8224, 64)
    # two workgroups share a unit's LDS: 4 bits have a table of 68 KB, one range of up to 6144 channels their activations, 12, and norms 64 bytes of their own
    assert makes(True, 4, half, 5632, 20480) and not makes(True, 4, half, 5664, 20480) and not makes(True, 4, half, 6144, 20480) and makes(False, 4, half, 6144, 15360)
    assert makes(False, 4, half, 17920, 5120) and not makes(False, 3, half, 28672, 8192) and not makes(True, 4, torch.float32, 4096, 4096)


def test_options_set_after_a_step_are_asked_for_again():
    """Fewer ranges of channels leave a product no room for its activations: what a layer was told before an option changed does not hold behind it."""
    from decdec_amd import _lib, decode_ops
    from decdec_amd.linear import SQLLMLinear, step_layer
    l = SQLLMLinear(14336, 4096, 4, dtype=torch.float16, device="cpu")
    room = torch.zeros(l.lut.numel() + 64, dtype=torch.float16)              # on the CPU a tensor may start anywhere
    first = (-room.data_ptr() % 16) // room.element_size()
    l._buffers["lut"], l.external_zero = room[first:first + l.lut.numel()].view(l.lut.shape), True
    ask = lambda: [step_layer(l, False, torch.float16, -1), decode_ops.product_makes(False, 4, torch.float16, 14336, 4096),
                   bool(_lib.load().decdec_sqllm_step_fuses(0, 4, 1, 14336, 4096))]
    with torch.no_grad():
        for name in ("gemv_max_k_ranges", "sqllm_ktiles"):
            assert ask() == [True] * 3
            _lib.set_option(name, 1)
            try:
                assert ask() == [False] * 3, name
            finally:
                _lib.set_option(name, 0)
        assert ask() == [True] * 3


def test_steps_of_other_layers_are_not_asked_about_their_products(monkeypatch):
    """Whether products make their activations is host work in every step that is not captured: layers of other kinds, and compensated ones, are told apart
    by what they are, without a look at a tensor or a module in between."""
    from decdec_amd import ext
    from decdec_amd.linear import APLinear, LUTGEMMLinear, SQLLMLinear
    from decdec_amd.model import ModelArgs, TransformerBlock

    def asked(*args):
        raise AssertionError("asked")
    monkeypatch.setattr(ext, "on_kernels", asked)
    h = torch.zeros(1, 1, 128, dtype=torch.float16)
    args = ModelArgs(n_layer=1, n_head=1, n_local_heads=1, dim=128, intermediate_size=256, vocab_size=16)
    for kind, more in ((APLinear, {}), (LUTGEMMLinear, {"group_size": 128}), (SQLLMLinear, {})):
        b = TransformerBlock(args, kind, {"bitwidth": 4, "dtype": torch.float16, "device": "cpu", **more})
        for l in b.dec_linears():
            l.external_zero, l.dec_config = True, 1 if kind is SQLLMLinear else None
        assert b._products_make(h, None) == (False, False, False)
    b.feed_forward.w2.dec_config = None
    with pytest.raises(AssertionError, match="asked"):
        b._products_make(h, None)


def test_a_norms_sum_goes_where_no_workgroup_reads():
    """The first workgroup of a product that norms its input writes the sum while the others read what it is made of: memory that overlaps is refused, ahead of a launch."""
    from decdec_amd import _lib
    K, N = 256, 64
    room = torch.zeros(8 * K, dtype=torch.float16)
    at = room.data_ptr() + -room.data_ptr() % 16
    x, y, w, out = at, at + 4 * K, at + 8 * K, at + 10 * K     # a gap behind x
    call = lambda h: _lib.load().decdec_sqllm_norm_gemv(x, y, w, 1e-5, h, out, at, at, 4, 1, K, N, None)
    for h in (x, y, w, x + 8, x + 2 * K - 8, y - 8, y + 2 * K - 8, w - 2 * K + 8):
        assert call(h) != 0 and "other workgroups" in _lib.last_error(), h - at
