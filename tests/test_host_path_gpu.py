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
