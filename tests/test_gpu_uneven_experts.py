"""Row tiles of 128 with uneven experts: tiles dealt to the XCDs by columns, and experts with second tiles dealt by their size.

16 experts of 3072 x 3072: both products have column tiles of 256 and of 128 rows, each a multiple of eight.  Float32 products of torch
on the same routing are the reference; the bounds are the layer's stated target (max-abs 2e-2, mean relative 1e-3 against float32:
fp16 activations between the products, 2^-12 relative each, averaged over 3072 of them)."""
import pytest
import torch

from electrock_infer_amd import fused_experts
from tests.gpu_util import DEV, announce, error_stats, gpu_inputs

pytestmark = pytest.mark.gpu
E, H, I = 16, 3072, 3072


@pytest.fixture(scope="module")
def weights():
    _, _, w13, w2 = gpu_inputs(1, H, I, E=E, seed=3)
    return w13, w2


def reference(x, logits, w13, w2):
    weight, chosen = torch.softmax(logits.float(), dim=-1).topk(2, dim=-1)
    weight = weight / weight.sum(dim=-1, keepdim=True)
    out = torch.zeros(x.shape[0], H, device=DEV)
    for e in range(E):
        t, k = (chosen == e).nonzero(as_tuple=True)
        gate, up = (x[t].float() @ w13[e].float().t()).chunk(2, dim=-1)
        out.index_add_(0, t, (torch.nn.functional.silu(gate) * up) @ w2[e].float().t() * weight[t, k, None])
    return out


# experts ahead of the others, by how much: dealt in their order (no or one second tile), by size (several, ties of 3 and 3), some
# and nearly all experts without rows; the last one ahead, the first one ahead
@pytest.mark.parametrize("ahead", [{}, {15: 1.5}, {0: 2.5}, {3: 3.0, 9: 3.0, 12: 2.0}, {5: 30.0, 6: 30.0}, {7: 30.0}])
@pytest.mark.parametrize("T", [65, 201, 352])
def test_uneven_experts(weights, T, ahead):
    announce(f"uneven experts T={T} ahead={ahead}")
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, H, generator=g, device=DEV).to(torch.bfloat16)
    logits = torch.randn(T, E, generator=g, device=DEV)
    for e, by in ahead.items():
        logits[:, e] += by
    logits = logits.to(torch.bfloat16)
    got = fused_experts(x, *weights, logits, 2, renormalize=True, out_dtype=torch.float32)
    st = error_stats(got, reference(x, logits, *weights))
    assert st["max_abs"] <= 2e-2 and st["mean_rel"] <= 1e-3, st
