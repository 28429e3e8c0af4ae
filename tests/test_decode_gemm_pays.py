"""Which decode-batch products go to the weight-streaming kernel and which to the library, and that both give them."""
import itertools

import pytest
import torch
import torch.nn.functional as F

from electrock_infer_amd import _lib
from electrock_infer_amd.layers import decoder_ops as ops
from tests.gpu_util import announce

F32, BF16 = _lib.DTYPE_F32, _lib.DTYPE_BF16


def test_routes():
    lib = _lib.load_decoder()
    pays = lib.ed_decode_gemm_pays
    # one tile and two of tokens on the projections of a layer, every form
    for T, (N, K) in itertools.product((1, 4, 16, 17, 32), ((2048, 2048), (6144, 2048), (4096, 4096), (8192, 4096), (32000, 2048), (32000, 4096))):
        assert pays(T, N, K, 0, BF16) and pays(T, N, K, 0, F32) and pays(T, N, K, 1, BF16) and pays(T, N // 2, K, 2, BF16)
    # few rows and a long sum, rows of 64 to a workgroup for a part of the chip, many tokens on large weights
    for T, N, K, act, dtype in ((64, 1024, 8192, 0, BF16), (40, 1024, 12288, 1, BF16), (40, 1024, 12288, 2, BF16), (48, 1024, 4096, 0, F32), (8, 4096, 16384, 0, BF16),
                                (24, 12288, 4096, 0, BF16), (32, 10240, 3072, 0, F32), (64, 8192, 4096, 0, BF16), (64, 32000, 4096, 0, BF16)):
        assert pays(T, N, K, act, dtype) == 0, (T, N, K, act)
    for T, N, K, act, dtype in ((0, 64, 64, 0, BF16), (65, 64, 64, 0, BF16), (4, 0, 64, 0, BF16), (4, 64, 100, 0, BF16), (4, 64, 64, 3, BF16), (4, 64, 64, 0, 7), (4, 1 << 30, 64, 2, 2)):
        assert pays(T, N, K, act, dtype) == 0
    assert all(lib.ed_decode_gemm_plain_pays(T, N, K) == pays(T, N, K, 0, BF16) for T, N, K in itertools.product((1, 20, 64, 65), (64, 1000, 12288), (64, 4096, 16384)))


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", [(64, 1024, 4160), (64, 1024, 4096), (33, 1024, 2112), (24, 9216, 2112), (16, 9216, 4160), (17, 10240, 2048), (49, 4096, 4096), (49, 4098, 4096), (8, 2050, 12352),
                                   (20, 3072, 8256)])
def test_both_sides_of_the_lines(T, N, K):
    announce(f"decode gemm routes {T} {N} {K}")
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    x, w = torch.randn(T, K, generator=g, device="cuda").bfloat16(), (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    want = x.double() @ w.double().t()
    off = lambda got, ref: float((got.double() - ref).norm() / ref.norm())
    # float32 sums; results, and the library's product in front of an activation, rounded to bf16: 2^-8 of a value
    assert off(ops.linear_f32(x, w), want) < 1e-5
    parts = ops.linear_parts(x, w, exact=True)
    assert off(parts.sum(0) if parts.dim() == 3 else parts, want) < 1e-5
    assert off(ops.linear(x, w), want) < 2.0 ** -8
    assert off(ops.linear(x, w, "relu_squared"), F.relu(want) ** 2) < 3 * 2.0 ** -8
    assert off(ops.linear_silu_gate(x, w), F.silu(want[:, :N // 2]) * want[:, N // 2:]) < 3 * 2.0 ** -8
