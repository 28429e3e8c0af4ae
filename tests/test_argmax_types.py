"""The greedy token of rows that its kernel does not take: the same places as the library's."""
import pytest
import torch

from electrock_infer_amd.layers.decoder_ops import argmax_rows
from tests.gpu_util import announce

TYPES = [torch.bfloat16, torch.float16, torch.float32, torch.float64, torch.int64]


def check(dtype, device):
    g = torch.Generator().manual_seed(1)
    for shape in ((7,), (3, 1001), (2, 3, 50), (0, 40), (4, 1)):
        x = (torch.randn(shape, generator=g) * 1000).to(dtype).to(device)
        got = argmax_rows(x)
        assert got.dtype == torch.int32 and got.shape == x.shape[:-1]
        assert torch.equal(x.gather(-1, got.long().unsqueeze(-1)).squeeze(-1), x.max(-1).values if x.numel() else x[..., 0])
    with pytest.raises((IndexError, RuntimeError)):
        argmax_rows(torch.zeros(3, 0, dtype=dtype, device=device))


@pytest.mark.parametrize("dtype", TYPES)
def test_host_rows(dtype):
    check(dtype, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", TYPES)
def test_device_rows(dtype):
    announce(f"argmax of {dtype}")
    check(dtype, "cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("T,V", [(1, 1 << 17), (1, (1 << 17) + 1), (2, (1 << 17) + 1), (1, 500001), ((1 << 22) - 1, 3), (1 << 22, 3)])
def test_long_rows_and_many(T, V):
    announce(f"argmax {T} x {V}")
    x = torch.randn(T, V, generator=torch.Generator(device="cuda").manual_seed(V), device="cuda")
    x[:, V // 2] = x[:, V - 1] = 9.0                           # the first of equal ones
    assert bool((argmax_rows(x) == V // 2).all())
