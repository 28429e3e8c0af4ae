"""The weight-streaming product of decode batches at the edges of its tiles and of the rule that picks them: the kernel itself into memory
that holds NaN, and the layers' functions, which take the tiled kernel or the library where those are faster."""
import pytest
import torch
import torch.nn.functional as F

from electrock_infer_amd import _lib
from electrock_infer_amd.layers import decoder_ops as ops
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def operands(T, N, K):
    g = torch.Generator().manual_seed(T * 7919 + N * 31 + K)
    x, w = torch.randn(T, K, generator=g).to(BF16), (torch.randn(N, K, generator=g) * K ** -0.5).to(BF16)
    return x.cuda(), w.cuda(), x.double() @ w.double().t()


def off(got, want):
    return float((got.double().cpu() - want).norm() / (want.norm() or 1.0))


# sums of K products of bf16 values in float32: about sqrt(K) 2^-24, far below 1e-5; a result rounded to bf16: no value is off by
# more than half a step, 2^-8 of it
F32_TOL, BF16_TOL = 1e-5, 2.0 ** -8 + 1e-5


def product(x, w, cols, splits=1, act=0, dtype=BF16):
    """The kernel itself, with a row behind the result that has to stay."""
    T, K = x.shape
    full = torch.full((splits * T + 1, cols), float("nan"), dtype=dtype, device="cuda")
    code = _lib.load_decoder().ed_decode_gemm(x.data_ptr(), w.data_ptr(), full.data_ptr(), _lib.dtype_code(dtype), splits, T, cols, K, act,
                                              _lib.current_stream(x.device))
    assert code == 0 and bool(full[-1].isnan().all())
    return full[:-1].view(splits, T, cols)


# Every form: tokens in ones to fours of 16; rows in ones (to 4096), twos (to 8192 or, up to 32 tokens, 9216), fours of eight waves (to 16384, from 33
# tokens) and of four waves, at their edges and with remainders; k: one step, fewer steps than waves, a range that waves share unevenly
@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(1, 64), (50, 192), (4096, 576), (4102, 128), (8192, 192), (8198, 64), (9216, 64), (9222, 128), (16384, 64), (16390, 192), (20000, 1088)])
def test_every_form_of_the_kernel(T, N, K):
    announce(f"decode gemm forms {T} {N} {K}")
    x, w, want = operands(T, N, K)
    assert off(product(x, w, N)[0], want) < BF16_TOL
    assert off(product(x, w, N, dtype=torch.float32)[0], want) < F32_TOL
    assert off(product(x, w, N, act=1)[0], F.relu(want) ** 2) < BF16_TOL
    if N % 2 == 0:
        half = N // 2
        assert off(product(x, w, half, act=2)[0], F.silu(want[:, :half]) * want[:, half:]) < BF16_TOL


# (rows in 32s and, from 33 tokens and 4096 rows on, in 64s where as many ranges fill the chip)
@pytest.mark.parametrize("T", [1, 17, 33, 64])
@pytest.mark.parametrize("N,K,splits", [(40, 8192, 8), (2048, 6144, 4), (4096, 1024, 2), (4130, 2048, 4), (4160, 4096, 3), (512, 1088, 17)])
def test_every_form_of_partial_sums(T, N, K, splits):
    announce(f"decode gemm forms of parts {T} {N} {K} {splits}")
    x, w, want = operands(T, N, K)
    assert off(product(x, w, N, splits, dtype=torch.float32).sum(0), want) < F32_TOL


# tokens: around every tile edge; rows: few, a remainder, as many as the rule takes to either kernel; k: one step, a range that waves share unevenly
@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 48, 49, 63, 64])
@pytest.mark.parametrize("N,K", [(1, 64), (50, 192), (4096, 128), (4100, 576), (8200, 64), (16400, 128)])
def test_products(T, N, K):
    announce(f"decode gemm {T} {N} {K}")
    x, w, want = operands(T, N, K)
    assert ops._skinny_splits(x, w) > 0
    assert off(ops.linear_f32(x, w), want) < F32_TOL
    assert off(ops.linear(x, w), want) < BF16_TOL
    assert off(ops.linear(x, w, "relu_squared"), F.relu(want) ** 2) < BF16_TOL
    if N % 2 == 0:
        half = N // 2
        assert off(ops.linear_silu_gate(x, w), F.silu(want[:, :half]) * want[:, half:]) < BF16_TOL


@pytest.mark.parametrize("T,N,K", [(1, 2048, 4096), (16, 40, 8192), (32, 4096, 1024), (48, 4096, 4096), (64, 4130, 1088), (64, 2048, 6144)])
def test_partial_sums(T, N, K):
    announce(f"decode gemm parts {T} {N} {K}")
    x, w, want = operands(T, N, K)
    parts = ops.linear_parts(x, w)
    assert parts.dim() == 3 and parts.shape[0] == ops._skinny_splits(x, w) > 1
    assert off(parts.sum(0), want) < F32_TOL
    # any number of ranges
    for splits in (2, 3, K // 64 if K // 64 <= 64 else 64):
        out = torch.full((splits, T, N), float("nan"), dtype=torch.float32, device="cuda")
        assert _lib.load_decoder().ed_decode_gemm(x.data_ptr(), w.data_ptr(), out.data_ptr(), _lib.DTYPE_F32, splits, T, N, K, 0,
                                                  _lib.current_stream(x.device)) == 0
        assert off(out.sum(0), want) < F32_TOL


def test_rows_that_lie_apart_go_to_the_library():
    """A view of wider rows, and operands off the kernel's alignment, as before."""
    announce("decode gemm strided weights")
    x, w, want = operands(20, 4096, 4608)
    wide = torch.cat([w, w], 1)[:, :4608]
    assert ops._skinny_splits(x, wide) == 0 and off(ops.linear(x, wide), want) < BF16_TOL
    shifted = torch.empty(20 * 4608 + 1, dtype=BF16, device="cuda")[1:].view(20, 4608).copy_(x)
    assert ops._skinny_splits(shifted, w) == 0 and off(ops.linear(shifted, w), want) < BF16_TOL


# rows in 64s and in 32s to a workgroup, by how many ranges K has room for
@pytest.mark.parametrize("T,N,K", [(33, 4096, 1024), (64, 4096, 1024), (48, 4096, 1536), (64, 4096, 1984), (64, 4096, 2048), (49, 4160, 1536), (64, 6144, 1024)])
def test_partial_sums_of_short_rows(T, N, K):
    test_partial_sums(T, N, K)
