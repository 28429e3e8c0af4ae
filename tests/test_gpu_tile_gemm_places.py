"""The tiled product of tokens that are alike: the same bits wherever they stand in the batch."""
import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce
from tests.test_gpu_tile_gemm import product

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


# row tiles of 64 and of 128 tokens, one and several, and the last of them ragged; ranges of K of one step, of several and whole
@pytest.mark.parametrize("T", [33, 65, 129, 300, 1030])
@pytest.mark.parametrize("N,K", [(256, 320), (1028, 832), (2048, 2048), (4099, 448)])
def test_equal_tokens(T, N, K):
    announce(f"tile gemm places {T} {N} {K}")
    g = torch.Generator(device="cuda").manual_seed(N + K)
    token, w = torch.randn(1, K, generator=g, device="cuda").to(BF16), (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    x = token.expand(T, K).contiguous()
    results = [product(x, w, N, act=act) for act in (0, 1)] + [product(x, w, N // 2, act=2)]
    results += [product(x, w, N, splits, dtype=torch.float32) for splits in (1, 2, K // 64)]
    for out in results:
        assert torch.equal(out, out[:, :1].expand_as(out))
