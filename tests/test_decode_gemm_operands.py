"""Which operands the decode-batch product takes: it reads dense rows from a 16-byte boundary, everything else is the library's."""
import pytest
import torch
import torch.nn.functional as F

from electrock_infer_amd.layers import decoder_ops as ops
from tests.gpu_util import announce

BF16 = torch.bfloat16
SIZES = [(1, 48, 64), (4, 4096, 4096), (16, 512, 1024), (32, 48, 192), (64, 2048, 2048)]


def forms(T, N, K, device):
    """(name, x, weight) of equal values: dense, rows that lie apart, columns that lie apart, either operand off its boundary."""
    g = torch.Generator().manual_seed(N + K)
    x, w = torch.randn(T, K, generator=g).to(BF16).to(device), (torch.randn(N, K, generator=g) * K ** -0.5).to(BF16).to(device)
    shifted = lambda t: torch.empty(t.numel() + 1, dtype=BF16, device=device)[1:].view(t.shape).copy_(t)
    yield "dense", x, w
    yield "rows of wider ones", x, torch.cat([w, -w], 1)[:, :K]
    yield "every other row", x, torch.stack([w, -w], 1).view(2 * N, K)[::2]
    yield "transposed", x, w.t().contiguous().t()
    yield "weights off a boundary", x, shifted(w)
    yield "tokens off a boundary", shifted(x), w
    if T > 1:
        yield "rows of wider tokens", torch.cat([x, -x], 1)[:, :K], w


@pytest.mark.parametrize("T,N,K", SIZES)
def test_only_dense_operands_are_taken(T, N, K):
    for name, x, w in forms(T, N, K, "cpu"):
        assert (ops._skinny_splits(x, w) > 0) == (name == "dense"), name


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", SIZES)
def test_every_form_gives_the_product(T, N, K):
    for name, x, w in forms(T, N, K, "cuda"):
        announce(f"decode gemm operands {T} {N} {K} {name}")
        want = x.double().cpu() @ w.double().cpu().t()
        # float32 sums of bf16 products; results (and a product in front of an activation) rounded to bf16, 2^-8 of a value
        off = lambda got, ref: float((got.double().cpu() - ref).norm() / ref.norm())
        assert off(ops.linear_f32(x, w), want) < 1e-5, name
        parts = ops.linear_parts(x, w)
        assert off(parts.sum(0) if parts.dim() == 3 else parts, want) < 2.0 ** -8, name
        assert off(ops.linear(x, w), want) < 2.0 ** -8, name
        assert off(ops.linear(x, w, "relu_squared"), F.relu(want) ** 2) < 3 * 2.0 ** -8, name
        gated = F.silu(want[:, :N // 2]) * want[:, N // 2:]
        assert off(ops.linear_silu_gate(x, w), gated) < 3 * 2.0 ** -8, name


def bf16(*shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(sum(shape))).to(BF16)


# (on the CPU: the product itself never runs on these)
@pytest.mark.parametrize("x,w", [(bf16(8, 128), bf16(48, 64)), (bf16(8, 64), bf16(48, 128)), (bf16(64, 4096), bf16(6144, 2048)), (bf16(8, 64), bf16(48, 64).float()),
                                 (bf16(8, 64).float(), bf16(48, 64)), (bf16(8, 64), bf16(48, 64).half())])
def test_operands_that_do_not_fit_are_refused(x, w):
    assert ops._skinny_splits(x, w) == 0
    for product in (ops.linear, ops.linear_parts, lambda x, w: ops.linear(x, w, "relu_squared"), ops.linear_silu_gate):
        with pytest.raises((RuntimeError, NotImplementedError)):
            product(x, w)


def test_operands_on_two_devices_are_not_taken():
    assert ops._skinny_splits(bf16(8, 64), torch.empty(48, 64, dtype=BF16, device="meta")) == 0


@pytest.mark.parametrize("shape", [(64,), (1, 64), (2, 3, 64), (64, 64, 64), (3, 1, 1, 64)])
def test_rows_of_any_shape_and_gradients_are_the_librarys(shape):
    x, w = bf16(*shape), bf16(48, 64)
    if len(shape) != 2:
        assert ops._skinny_splits(x, w) == 0 and torch.equal(ops.linear(x, w), F.linear(x, w))
    x.requires_grad_()
    assert ops._skinny_splits(x, w) == 0
    ops.linear(x, w).sum().backward()
    # (sums of 48 standard normal values, about 20 at most, rounded to bf16)
    assert float((x.grad - w.float().sum(0)).abs().max()) < 20 * 2.0 ** -8
    if len(shape) == 2:
        with torch.no_grad():
            assert ops._skinny_splits(x, w) > 0


def test_mapped_forward_differentiated_and_traced_calls_are_the_librarys():
    x, w, t = bf16(3, 8, 64), bf16(48, 64), bf16(8, 64)
    assert torch.equal(torch.func.vmap(lambda a: ops.linear(a, w))(x), torch.func.vmap(lambda a: F.linear(a, w))(x))
    product = lambda f: torch.func.jvp(lambda a: f(a, w), (x[0],), (t,))
    assert all(torch.equal(a, b) for a, b in zip(product(ops.linear), product(F.linear)))
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x[0], t)
        assert ops._skinny_splits(dual, w) == 0
        assert torch.equal(torch.autograd.forward_ad.unpack_dual(ops.linear(dual, w)).tangent, F.linear(t, w))
    with torch.no_grad():
        traced = torch.jit.trace(lambda a: ops.linear(a, w), x[0], check_trace=False)
        assert torch.equal(traced(x[1]), F.linear(x[1], w)) and ops._skinny_splits(x[0], w) > 0


@pytest.mark.parametrize("T,N,K", SIZES + [(20, 4608, 4096)])
def test_host_tensors_are_the_librarys(T, N, K):
    x, w = bf16(T, K), bf16(N, K)
    want = F.linear(x, w)
    assert torch.equal(ops.linear(x, w), want) and torch.equal(ops.linear_parts(x, w), want)
