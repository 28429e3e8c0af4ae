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
