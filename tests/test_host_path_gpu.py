"""Native host path of the eager operators (csrc/host): the same results as the torch.library route bit for bit (it launches
the same kernels), and NotImplemented, without a launch, for every call that route has to see."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _int4(n, k, g=64):
    from ao_amd import ops

    w = (torch.randn(n, k, generator=torch.Generator().manual_seed(n + k)) * 0.02).bfloat16().cuda()
    return ops.int4wo_quantize_pack(w, g)


@pytest.mark.parametrize("shape", [(1, 256, 48), (16, 4096, 4096), (33, 1024, 272), (65, 384, 128)])
@pytest.mark.parametrize("bias", [False, True])
def test_int4_linear_is_the_operator(shape, bias):
    from ao_amd import ops

    m, k, n = shape
    packed, qparams = _int4(n, k)
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    b = torch.randn(n, device="cuda", dtype=torch.bfloat16) if bias else None
    want = torch.ops.torchao.int4wo_linear.default(x, packed, qparams, 64, n, b, False)
    got = ops.host.int4wo_linear(x, packed, qparams, 64, n, k, b, None)
    assert torch.equal(got, want)
    if m == 16:  # leading dimensions are kept
        got = ops.host.int4wo_linear(x.view(2, 8, k), packed, qparams, 64, n, k, b, None)
        assert got.shape == (2, 8, n) and torch.equal(got.view(m, n), want)


def test_module_call_takes_the_host_path(monkeypatch):
    """F.linear of every weight class reaches the host functions; the result is the torch.library operator's."""
    import ao_amd
    from ao_amd import ops

    for recipe, name, dtype in ((ao_amd.int4_weight_only(64), "int4wo_linear", torch.bfloat16),
                                (ao_amd.int8_weight_only(), "int8wo_linear", torch.bfloat16),
                                (ao_amd.fp6_llm_weight_only(), "fp6_linear", torch.float16)):
        lin = torch.nn.Linear(512, 256, bias=True, device="cuda", dtype=dtype)
        ao_amd.quantize_(lin, recipe)
        x = torch.randn(3, 5, 512, device="cuda", dtype=dtype)
        seen, native = [], getattr(ops.host, name)
        monkeypatch.setattr(ops.host, name, lambda *a: seen.append(native(*a)) or seen[-1])
        with torch.no_grad():
            got = lin(x)
            assert seen and torch.is_tensor(seen[-1]) and got.shape == (3, 5, 256)
            monkeypatch.setattr(ops.host, name, lambda *a: NotImplemented)
            assert torch.equal(lin(x), got)
        monkeypatch.setattr(ops.host, name, native)
        y = lin(x.clone().requires_grad_())  # a gradient to record: left to torch.library
        assert y.shape == got.shape


def test_calls_that_others_have_to_see_are_declined():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from ao_amd import ops

    n, k = 64, 256
    packed, qparams = _int4(n, k)
    x = torch.randn(2, k, device="cuda", dtype=torch.bfloat16)

    def call(x=x, packed=packed, k=k, bias=None):
        return ops.host.int4wo_linear(x, packed, qparams, 64, n, k, bias, None)

    assert torch.is_tensor(call())

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatches(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (Functions(), Dispatches(), FakeTensorMode()):
        with mode:
            assert call() is NotImplemented
    assert call(x=x.clone().requires_grad_()) is NotImplemented
    assert call(x=x.float()) is NotImplemented
    assert call(x=x.cpu()) is NotImplemented
    assert call(x=x.t().contiguous().t()) is NotImplemented
    assert call(x=x[:, :128]) is NotImplemented          # another K
    assert call(k=128) is NotImplemented
    assert call(packed=packed[:2]) is NotImplemented      # fewer row blocks than N asks for
    assert call(bias=torch.zeros(n - 1, device="cuda", dtype=torch.bfloat16)) is NotImplemented
    assert torch.func.vmap(lambda r: torch.tensor(call(x=r[None]) is NotImplemented))(x).all()


def _plain_calls():
    """(function, arguments, index of the activations) of a call that each function serves."""
    import ao_amd
    from ao_amd import ops
    from ao_amd._models.llama.generate import build_random_model
    from ao_amd.prototype.hqq.mixed_mm import pack_2xint4

    def weight(recipe, dtype):
        lin = torch.nn.Linear(256, 256, bias=False, device="cuda", dtype=dtype)
        ao_amd.quantize_(lin, recipe)
        return lin.weight

    def x(dtype):
        return torch.randn(2, 256, device="cuda", dtype=dtype)

    w8, w6 = weight(ao_amd.int8_weight_only(), torch.bfloat16), weight(ao_amd.fp6_llm_weight_only(), torch.float16)
    codes = pack_2xint4(torch.randint(0, 16, (256, 256), dtype=torch.uint8, device="cuda"))
    q = [torch.rand(4, 256, device="cuda", dtype=torch.bfloat16) for _ in range(2)]
    model = build_random_model("tiny128", torch.device("cuda"), "int4wo-64")
    model.setup_caches(1, 64)
    rows = torch.randn(1, 5, 512, device="cuda", dtype=torch.bfloat16)
    packed, qparams = _int4(64, 256)
    return {
        "int4wo_linear": ([x(torch.bfloat16), packed, qparams, 64, 64, 256, None, None], 0),
        "int8wo_linear": ([x(torch.bfloat16), w8.layout_tensor.int_data, w8.layout_tensor.scale, None, None], 0),
        "fp6_linear": ([3, 2, x(torch.float16), w6.native(), w6.scale], 2),
        "hqq_mixed_mm": ([x(torch.bfloat16), codes, *q, 64, False], 0),
        "llama_forward": ([model._host_plan("int4", 5), rows, None, torch.arange(5, device="cuda")], 1),
    }


@pytest.mark.parametrize("name", ["int4wo_linear", "int8wo_linear", "fp6_linear", "hqq_mixed_mm", "llama_forward"])
def test_every_function_declines_what_others_have_to_see(name):
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from ao_amd import ops

    args, i = _plain_calls()[name]

    def call(x=args[i]):
        return getattr(ops.host, name)(*args[:i], x, *args[i + 1:])

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatches(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Subclass(torch.Tensor):
        pass

    with torch.no_grad():
        assert torch.is_tensor(call())
        for mode in (Functions(), Dispatches(), FakeTensorMode()):
            with mode:
                assert call() is NotImplemented
        x = args[i]
        with forward_ad.dual_level():
            assert call(forward_ad.make_dual(x, x)) is NotImplemented
        assert torch.func.vmap(lambda r: torch.tensor(call(r) is NotImplemented))(x[None]).all()
        for other in (x.cpu(), x.float(), x.transpose(-1, -2), x.as_subclass(Subclass), x[..., :128], None, 3):
            assert call(other) is NotImplemented
    if name != "llama_forward":  # its norms are parameters that ask for a gradient
        assert torch.is_tensor(call())
    assert call(x.clone().requires_grad_()) is NotImplemented


def test_hqq_flag_that_is_not_a_bool():
    """The operator takes a number for `transposed`; on a square weight the other product has the same shape."""
    from ao_amd import ops

    (x, codes, scales, zeros, group, _), _ = _plain_calls()["hqq_mixed_mm"]
    want = [ops.hqq_mixed_mm_mfma(x, codes, scales, zeros, group, t) for t in (False, True)]
    assert not torch.equal(*want)
    for flag in (0, 1):
        assert torch.equal(ops.hqq_mixed_mm_mfma(x, codes, scales, zeros, group, flag), want[flag])
