"""Products that somebody watches, records or changes are the library's for decode batches and prompts alike: under a tracer, a compiler,
fake tensors, a mode, a subclass or a cast a C call would be lost, or reach the kernel without an address.

On the CPU: tensors pass as the GPU's and the C calls fail the test, so only the operands' check stands between the two."""
import pytest
import torch
import torch.nn.functional as F
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from electrock_infer_amd.layers import decoder_ops as ops

BF16 = torch.bfloat16
PRODUCTS = [ops.linear, ops.linear_parts]


class Called(Exception):
    pass


@pytest.fixture(params=[8, 300], ids=["decode", "prompt"])
def operands(request, monkeypatch):
    def called(*args):
        raise Called
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda t: True), raising=False)
    monkeypatch.setattr(ops, "_tile_gemm", called)
    monkeypatch.setattr(ops, "_decode_gemm", called)
    g = torch.Generator().manual_seed(request.param)
    x, w = torch.randn(request.param, 1024, generator=g).to(BF16), torch.randn(2048, 1024, generator=g).to(BF16)
    with torch.no_grad():
        for product in PRODUCTS[:1]:
            with pytest.raises(Called):          # (nobody watches: the package's kernels take it)
                product(x, w)
        yield x, w


@pytest.mark.parametrize("product", PRODUCTS)
def test_recorded(operands, product):
    x, w = operands
    graph = make_fx(lambda a: product(a, w))(x)
    names = [str(n.target) for n in graph.graph.nodes if n.op == "call_function"]
    assert any("mm" in n or "linear" in n for n in names), names
    assert torch.equal(graph(-x), F.linear(-x, w))


@pytest.mark.parametrize("product", PRODUCTS)
def test_fake_tensors(operands, product):
    x, w = operands
    with FakeTensorMode() as mode:
        fake = mode.from_tensor(x), mode.from_tensor(w)
        assert product(*fake).shape == (x.shape[0], 2048)
    assert product(*fake).shape == (x.shape[0], 2048)          # (outside of their mode as well)


@pytest.mark.parametrize("product", PRODUCTS)
def test_compiled(operands, product):
    x, w = operands
    torch._dynamo.reset()
    assert torch.equal(torch.compile(lambda a, b: product(a, b), fullgraph=True, backend="eager")(x, w), F.linear(x, w))


@pytest.mark.parametrize("product", PRODUCTS)
def test_modes_and_subclasses(operands, product):
    x, w = operands
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Named(torch.Tensor):
        pass

    with Dispatch():
        got = product(x, w)
    assert torch.equal(got, F.linear(x, w)) and any("mm" in s for s in seen)
    with Function():
        got = product(x, w)
    assert torch.equal(got, F.linear(x, w)) and F.linear in seen
    assert type(product(x.as_subclass(Named), w)) is Named
    with torch.device("cpu"), pytest.raises(Called):           # (a default device changes no product)
        ops.linear(x, w)


@pytest.mark.parametrize("product", PRODUCTS)
def test_casts(operands, product):
    x, w = operands
    with torch.autocast("cpu", dtype=torch.float16):
        assert product(x, w).dtype == torch.float16
    with torch.autocast("cpu", dtype=BF16), pytest.raises(Called):
        ops.linear(x, w)
    with pytest.raises(Called):
        ops.linear(x, torch.nn.Parameter(w, requires_grad=False))
