"""The native pass of the Llama model (csrc/host/llama.cpp) against the module chain that it stands for: where the modules would
give something else it has to leave the prompt to them, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

RECIPES = ("int4", "int8", "fp6")


def _model(fmt, layers=2, intermediate=1024, positions=160, block_size=512, seed=0, heads=(4, 2), group=64):
    from ao_amd import fp6_llm_weight_only, int4_weight_only, int8_weight_only, quantize_
    from ao_amd._models.llama.generate import random_init_
    from ao_amd._models.llama.model import ModelArgs, Transformer

    args = ModelArgs(block_size=block_size, n_layer=layers, n_head=heads[0], n_local_heads=heads[1], dim=128 * heads[0],
                     intermediate_size=intermediate, vocab_size=1024)
    with torch.device("cuda"):
        model = Transformer(args).to(torch.bfloat16)
    random_init_(model, seed=seed)
    model = model.eval().to(torch.float16 if fmt == "fp6" else torch.bfloat16)
    quantize_(model, {"int4": lambda: int4_weight_only(group), "int8": int8_weight_only, "fp6": fp6_llm_weight_only}[fmt]())
    model.setup_caches(1, positions)
    return model


def _prompt(model, T, seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(0, model.config.vocab_size, (1, T), device="cuda", generator=g), torch.arange(T, device="cuda")


def _caches(model):
    return [c for b in model.layers for c in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache)]


def _both(model, tokens, pos):
    """(logits, caches) of the call as it is, and of the module chain."""
    runs = []
    for fused in (True, False):
        for c in _caches(model):
            c.zero_()
        model.use_fused_decode = fused
        with torch.no_grad():
            runs.append([model(tokens, pos)] + [c.clone() for c in _caches(model)])
    model.use_fused_decode = True
    return runs


def _same(got, want):
    return all(a.dtype is b.dtype and torch.equal(a, b) for a, b in zip(got, want))


# 1536 and 1537 rows: w1 and w3 go through a 16-bit copy of the weight and the library product, which autocast would cast
@pytest.mark.parametrize("fmt,T,intermediate", [(f, 17, 1024) for f in RECIPES] + [("int8", 1536, 8192), ("fp6", 1537, 8192)])
def test_autocast_prompts_run_as_modules(fmt, T, intermediate):
    model = _model(fmt, 1, intermediate, T, 2048)
    with torch.autocast("cuda", dtype=torch.bfloat16 if fmt == "fp6" else torch.float16):
        got, want = _both(model, *_prompt(model, T))
    assert _same(got, want) and not want[0].isnan().any()


class _Adapter(torch.nn.Linear):
    def forward(self, x):
        return super().forward(x) + x.mean(-1, keepdim=True)


class _Block(torch.nn.Module):
    def forward(self, x, input_pos, freqs_cis, mask):
        return x * 2


class _Cache(torch.nn.Module):
    """A cache of its own that stores halved values."""

    def __init__(self, like):
        super().__init__()
        self.k_cache, self.v_cache = like.k_cache, like.v_cache

    def update(self, input_pos, k, v):
        self.k_cache[:, :, input_pos], self.v_cache[:, :, input_pos] = k / 2, v / 2
        return self.k_cache, self.v_cache


def _adapt(linear):
    linear.__class__ = _Adapter


def _patch(module):
    forward = module.forward
    module.forward = lambda *a: forward(*a) * 2


def _layer_norm(module, name):
    setattr(module, name, torch.nn.LayerNorm(512, device="cuda", dtype=torch.bfloat16))


CHANGES = {
    "adapter in wqkv": lambda m, mp: _adapt(m.layers[1].attention.wqkv),
    "adapter in w2": lambda m, mp: _adapt(m.layers[0].feed_forward.w2),
    "adapter in output": lambda m, mp: _adapt(m.output),
    "patched linear": lambda m, mp: _patch(m.layers[0].feed_forward.w1),
    "patched feed-forward": lambda m, mp: _patch(m.layers[1].feed_forward),
    "patched class": lambda m, mp: mp.setattr(type(m.norm), "forward", lambda self, x: x * 2),
    "patched attention function": lambda m, mp: mp.setattr(torch.nn.functional, "scaled_dot_product_attention", lambda q, k, v, **kw: q * 2),
    "other norm in a block": lambda m, mp: _layer_norm(m.layers[0], "ffn_norm"),
    "other norm at the end": lambda m, mp: _layer_norm(m, "norm"),
    "other mask": lambda m, mp: setattr(m, "causal_mask", torch.ones_like(m.causal_mask)),
    "mask changed in place": lambda m, mp: m.causal_mask.fill_(True),
    "other block": lambda m, mp: m.layers.__setitem__(0, _Block()),
    "other cache": lambda m, mp: setattr(m.layers[0].attention, "kv_cache", _Cache(m.layers[0].attention.kv_cache)),
}


@pytest.mark.parametrize("change", list(CHANGES))
def test_changed_modules_run_as_modules(change, monkeypatch):
    """A module that is not the plain one is called: the prompt gives what the module chain gives."""
    model = _model("int4")
    CHANGES[change](model, monkeypatch)
    if change == "other block":  # the first block holds no cache any more
        with torch.no_grad():
            got = [model(*_prompt(model, 17))]
            model.use_fused_decode = False
            want = [model(*_prompt(model, 17))]
    else:
        got, want = _both(model, *_prompt(model, 17))
    assert _same(got, want)


@pytest.mark.parametrize("fmt", RECIPES)
def test_plain_prompts_take_the_native_pass(fmt, monkeypatch):
    from ao_amd import ops

    seen, native = [], ops.host.llama_forward
    monkeypatch.setattr(ops.host, "llama_forward", lambda *a: seen.append(native(*a)) or seen[-1])
    model = _model(fmt)
    with torch.no_grad():
        out = model(*_prompt(model, 17))
    assert len(seen) == 1 and seen[0] is out


def test_caches_made_in_inference_mode_take_the_native_pass(monkeypatch):
    from ao_amd import ops

    model = _model("int4", positions=32)
    seen, native = [], ops.host.llama_forward
    monkeypatch.setattr(ops.host, "llama_forward", lambda *a: seen.append(native(*a)) or seen[-1])
    with torch.inference_mode():
        model.setup_caches(1, 160)
        model(*_prompt(model, 17))
        assert torch.is_tensor(seen[-1])
        model.causal_mask[3, 9] = True
        model(*_prompt(model, 17))
    assert len(seen) == 1


@pytest.mark.parametrize("fmt", ["int4", "int8"])
def test_parametrized_weights_run(fmt):
    """Weights that are no entries of _parameters any more: plain tensors that a parametrization puts together again."""
    from ao_amd.utils import unwrap_tensor_subclass

    model, plain = _model(fmt), _model(fmt)
    unwrap_tensor_subclass(model)
    assert "weight" not in model.output._parameters
    assert _same(*_both(model, *_prompt(model, 17)))
    step = torch.tensor([[3]], device="cuda"), torch.tensor([17], device="cuda")
    with torch.no_grad():
        for m in (model, plain):
            for c in _caches(m):
                c.fill_(0.5)
        assert torch.equal(model(*step), plain(*step))


class _Table(torch.nn.Module):
    def __init__(self, like):
        super().__init__()
        self.table, self.calls = like.weight, 0

    def forward(self, idx):
        self.calls += 1
        return torch.nn.functional.embedding(idx, self.table) * 2


@pytest.mark.parametrize("fmt", RECIPES)
@pytest.mark.parametrize("kind", ["hook", "weight", "no weight"])
def test_the_embedding_module_is_called(fmt, kind):
    """Once for a prompt or a decode step, whatever module it is: it refuses tokens outside its table."""
    model, plain = _model(fmt), _model(fmt)
    with torch.no_grad():
        plain.tok_embeddings.weight.mul_(2)
    seen = []
    if kind == "hook":
        model.tok_embeddings.register_forward_hook(lambda m, i, o: seen.append(1) or o * 2)
    else:
        model.tok_embeddings = table = _Table(model.tok_embeddings)
        if kind == "weight":
            table.weight = table.table
    with torch.no_grad():
        for call in (_prompt(model, 17), (torch.tensor([[3]], device="cuda"), torch.tensor([17], device="cuda"))):
            if kind == "no weight":  # nothing says the type of the model: modules
                plain.use_fused_decode = False
            assert torch.equal(model(*call), plain(*call))
    assert (len(seen) if kind == "hook" else table.calls) == 2


@pytest.mark.parametrize("fmt", ["int4", "fp6"])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_negative_positions_count_from_the_end(fmt, dtype):
    """As indexing has it: from the end of the cache for the row, from the end of the rotary table for the angle.  Both paths take the
    same steps with sums in another order (3e-2 as for the decode steps; the caches of the first layer see one linear: 2^-8)."""
    model = _model(fmt)
    tokens, _ = _prompt(model, 5)
    got, want = _both(model, tokens, torch.tensor([3, -1, 7, -160, 159 - 64], device="cuda", dtype=dtype))
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a.float() - b.float()).norm() <= (3e-2 if i in (0, 3, 4) else 2 ** -8) * b.float().norm()
        assert torch.equal(a == 0, b == 0) if i in (1, 2) else not a.isnan().any()


def test_prompts_pass_the_range_checks_of_indexing():
    """Tokens go through torch's embedding kernel and positions through its indexing, which refuse what is out of range."""
    model = _model("int8")
    call = _prompt(model, 9)
    with torch.no_grad(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        model(*call)
    count = {e.key: e.count for e in prof.key_averages()}
    assert count.get("aten::embedding") == 1 and count.get("aten::index") == 1
    assert not any(k.startswith("torchao::") for k in count)  # the native pass, not the modules


def _call(name, *args):
    from ao_amd import _lib

    args = [a.data_ptr() if torch.is_tensor(a) else a for a in args]
    _lib.check(getattr(_lib.lib(), name)(*args, _lib.current_stream(torch.device("cuda"))))


def _linear(lin, x):
    w, op = lin.weight, torch.ops.torchao
    if hasattr(w, "fpx_data"):
        return op.fp6_linear_native.default(w.ebits, w.mbits, x, w.native(), w.scale)
    lay = w.layout_tensor
    if hasattr(lay, "packed_weight"):
        return op.int4wo_linear.default(x, lay.packed_weight, lay.scale_and_zero, lay.group_size, lay.N, None, False)
    return op.int8wo_linear.default(x, lay.int_data, lay.scale, None, False)


def _composed(model, tokens, pos):
    """The prompt kernel by kernel: logits and caches."""
    cfg, T = model.config, tokens.numel()
    f16 = int(model.freqs_cis.dtype is torch.float16)
    x = model.tok_embeddings(tokens).view(T, -1)
    n = torch.empty_like(x)
    blocks = list(model.layers)
    _call("ao_amd_rmsnorm_f16" if f16 else "ao_amd_rmsnorm_bf16", x, blocks[0].attention_norm.weight, T, cfg.dim, cfg.norm_eps, n)
    for b, after in zip(blocks, [b.attention_norm for b in blocks[1:]] + [model.norm]):
        kv, y = b.attention.kv_cache, torch.empty_like(x)
        _call("ao_amd_llama_prefill_attention", _linear(b.attention.wqkv, n), f16, model.freqs_cis, pos, 1, T, kv.k_cache, kv.v_cache,
              cfg.n_head, cfg.n_local_heads, 128, model.max_seq_length, y)
        h, hn = torch.empty_like(x), torch.empty_like(x)
        _call("ao_amd_add_rmsnorm", x, _linear(b.attention.wo, y), b.ffn_norm.weight, f16, T, cfg.dim, cfg.norm_eps, h, hn)
        gate, up = _linear(b.feed_forward.w1, hn), _linear(b.feed_forward.w3, hn)
        _call("ao_amd_silu_mul", gate, up, f16, gate.numel(), gate)
        x, n = torch.empty_like(x), torch.empty_like(x)
        _call("ao_amd_add_rmsnorm", h, _linear(b.feed_forward.w2, gate), after.weight, f16, T, cfg.dim, cfg.norm_eps, x, n)
    return [_linear(model.output, n).view(1, T, -1)] + [c.clone() for c in _caches(model)]


# Short prompts on every kind of product, and the lengths at which the weight goes through a 16-bit copy and the library product.
# 1088 and 2112 in_features, and 640 in groups of 256, end before the packed width.
@pytest.mark.parametrize("fmt,T,intermediate,heads,group", [(f, T, 1024, (4, 2), 64) for f in RECIPES for T in (2, 17, 33, 130)] +
                         [("int4", T, 1088, (4, 1), 64) for T in (17, 130)] +
                         [("int4", 4096, 2048, (4, 2), 64), ("int4", 4096, 2112, (5, 1), 256), ("int8", 1536, 8192, (4, 2), 0),
                          ("fp6", 1537, 8192, (4, 2), 0)])
def test_native_pass_is_its_kernels(fmt, T, intermediate, heads, group, monkeypatch):
    """Bit for bit the operators and kernels it is made of, each of which has a test of its own: no rounding, operand or route differs."""
    from ao_amd import ops

    model = _model(fmt, 2, intermediate, max(T, 160), 4096, 0, heads, group)
    tokens, pos = _prompt(model, T)
    seen, native = [], ops.host.llama_forward
    monkeypatch.setattr(ops.host, "llama_forward", lambda plan, *a: seen.append(plan) or native(plan, *a))
    with torch.no_grad():
        got = [model(tokens, pos)] + [c.clone() for c in _caches(model)]
        for c in _caches(model):
            c.zero_()
        want = _composed(model, tokens, pos)
    assert _same(got, want) and not want[0].isnan().any()
    (plan,) = seen
    two_pass = [lin[4] for layer in plan[8] for lin in layer if isinstance(lin, tuple)]
    assert any(two_pass) == (T >= 1536)


@pytest.mark.parametrize("fmt", RECIPES)
def test_prompts_in_a_captured_graph(fmt):
    """Replays on other tokens and positions, eager work in between, against eager calls."""
    model = _model(fmt)
    tokens, pos = _prompt(model, 33)
    static = tokens.clone(), pos.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.no_grad():
        model(*static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        logits = model(*static)
    for i in range(4):
        tokens, _ = _prompt(model, 33, 10 + i)
        with torch.no_grad():
            want = model(tokens, pos + 20 * i).clone()
            caches = [c.clone() for c in _caches(model)]
            for c in _caches(model):
                c.zero_()
            model(*_prompt(model, 20 * i)) if i else None
        static[0].copy_(tokens)
        static[1].copy_(pos + 20 * i)
        for c, w in zip(_caches(model), caches):
            c.copy_(w)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(logits, want) and all(map(torch.equal, _caches(model), caches))


@pytest.mark.parametrize("how", ["deepcopy", "file"])
def test_copies_of_a_model_take_the_native_pass(how, monkeypatch, tmp_path):
    """Unless their mask had been changed before."""
    import copy

    from ao_amd import ops

    def copied(model):
        if how == "deepcopy":
            return copy.deepcopy(model)
        torch.save(model, tmp_path / "model.pt")
        return torch.load(tmp_path / "model.pt", weights_only=False)

    model = _model("int8")
    seen, native = [], ops.host.llama_forward
    monkeypatch.setattr(ops.host, "llama_forward", lambda *a: seen.append(native(*a)) or seen[-1])
    want = _both(model, *_prompt(model, 17))[0]
    assert _same(_both(copied(model), *_prompt(model, 17))[0], want) and len(seen) == 2 and all(map(torch.is_tensor, seen))
    model.causal_mask.fill_(True)
    assert _same(*_both(copied(model), *_prompt(model, 17))) and len(seen) == 2
