"""The tiled product of decode batches and short prompts at the edges of its tiles, of its ring and of the rule that takes calls to it."""
import pytest
import torch
import torch.nn.functional as F

from electrock_infer_amd import _lib
from electrock_infer_amd.layers import decoder_ops as ops
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
# sums of K products of bf16 values in float32: about sqrt(K) 2^-24, far below 1e-5; a result rounded to bf16: no value is off by
# more than half a step, 2^-8 of it
F32_TOL, BF16_TOL = 1e-5, 2.0 ** -8 + 1e-5


def operands(T, N, K, x_stride=None, w_stride=None):
    g = torch.Generator().manual_seed(T * 7919 + N * 31 + K)
    x, w = torch.randn(T, x_stride or K, generator=g).to(BF16), (torch.randn(N, w_stride or K, generator=g) * K ** -0.5).to(BF16)
    x, w = x.cuda()[:, :K], w.cuda()[:, :K]
    return x, w, x.cpu().double() @ w.cpu().double().t()


def off(got, want):
    return float((got.double().cpu() - want).norm() / (want.norm() or 1.0))


def close(got, want, sums):
    """Every value of a bf16 result: half a step of its own (2^-8 of it), and what its float32 sums are off by, 1e-5 of ``sums``."""
    return bool(((got.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * sums).all())


def product(x, w, cols, splits=1, act=0, dtype=BF16):
    """The kernel itself, into memory that holds NaN, with a row behind the result that has to stay."""
    T, K = x.shape
    full = torch.full((splits * T + 1, cols), float("nan"), dtype=dtype, device="cuda")
    code = _lib.load_decoder().ed_tile_gemm(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), full.data_ptr(), _lib.dtype_code(dtype),
                                            splits, T, cols, K, act, _lib.current_stream(x.device))
    assert code == 0 and bool(full[-1].isnan().all())
    return full[:-1].view(splits, T, cols)


# rows around the tiles' edges; columns of one tile, remainders of 16 and of 4; K of one step, fewer than a ring, more than the
# deepest; enough columns for every form of a decode batch
@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 63, 64, 65, 127, 129, 300, 1030])
@pytest.mark.parametrize("N,K", [(34, 64), (70, 128), (1028, 320), (2056, 448), (4099, 832), (12290, 832), (20000, 192)])
def test_products(T, N, K):
    announce(f"tile gemm {T} {N} {K}")
    x, w, want = operands(T, N, K)
    # (a value of x w^T is of size one; u^2 and silu(g) u are off by their slopes times the sums' error, |u| and |g| below 8)
    assert close(product(x, w, N)[0], want, 1.0)
    got = product(x, w, N, dtype=torch.float32)[0].double().cpu()
    assert off(got, want) < F32_TOL and float((got - want).abs().max()) < 1e-4
    assert close(product(x, w, N, act=1)[0], F.relu(want) ** 2, 16.0)
    half = N // 2
    assert close(product(x, w, half, act=2)[0], F.silu(want[:, :half]) * want[:, half:2 * half], 16.0)
    for splits in {1, 2, 3, K // 64}:
        if splits <= K // 64:
            assert off(product(x, w, N, splits, dtype=torch.float32).sum(0), want) < F32_TOL


@pytest.mark.parametrize("T,N,K,x_stride,w_stride", [(200, 1100, 512, 576, 512), (1100, 200, 512, 512, 576), (130, 96, 128, 4096, 136)])
def test_rows_that_lie_apart(T, N, K, x_stride, w_stride):
    announce(f"tile gemm rows apart {T} {N} {K}")
    x, w, want = operands(T, N, K, x_stride, w_stride)
    assert off(product(x, w, N)[0], want) < BF16_TOL


@pytest.mark.parametrize("T,N,K", [(65, 1024, 512), (300, 2048, 2048), (300, 2048, 6144), (512, 4096, 4096), (1024, 2048, 4096), (513, 4096, 4096),
                                   (64, 2048, 2048), (64, 12288, 1024), (23, 6720, 1088), (16, 10240, 1024), (1, 8512, 2048), (300, 1000, 512), (300, 2048, 2056), (700, 6144, 2048)])
def test_every_route_gives_the_product(T, N, K):
    """What the rule takes and what it leaves to the library."""
    announce(f"tile gemm routes {T} {N} {K}")
    x, w, want = operands(T, N, K)
    parts, lib = ops.linear_parts(x, w), _lib.load_decoder()
    splits = lib.ed_tile_gemm_splits(T, N, K)
    if splits > 0:
        assert parts.dim() == (3 if splits > 1 else 2)
    assert off(parts.sum(0) if parts.dim() == 3 else parts, want) < BF16_TOL
    exact = ops.linear_parts(x, w, exact=True)
    assert exact.dtype == torch.float32 and off(exact.sum(0) if exact.dim() == 3 else exact, want) < F32_TOL
    assert off(ops.linear_f32(x, w), want) < F32_TOL
    assert off(ops.linear(x, w), want) < BF16_TOL
    # (behind the library's product the activation rounds once more, a squared value's error doubles)
    assert off(ops.linear(x, w, "relu_squared"), F.relu(want) ** 2) < 3 * BF16_TOL
    assert off(ops.linear_silu_gate(x, w), F.silu(want[:, :N // 2]) * want[:, N // 2:]) < 3 * BF16_TOL
    # operands off the kernel's boundaries are the library's
    wide = torch.cat([x, x[:, :4]], 1)[:, :K]
    shifted = torch.empty(N * K + 1, dtype=BF16, device="cuda")[1:].view(N, K).copy_(w)
    assert not ops._tiles_fit(wide, w) and not ops._tiles_fit(x, shifted) and not ops._fits(x, shifted)
    assert off(ops.linear(wide, w), want) < BF16_TOL and off(ops.linear(x, shifted), want) < BF16_TOL
