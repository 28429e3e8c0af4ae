"""Rows of a prompt in front of attention: the wave-per-token kernels against the general ones, which take the same tokens in smaller calls."""
import itertools

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
BF16, FEW = torch.bfloat16, 100            # (calls of so few tokens take the general kernels)


def values(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(BF16).cuda()


def same(got, want):
    """The two kernels add a row's squares up in another order: float32 results a few units apart, and so now and then another bf16."""
    a, b = got.float(), want.float()
    assert bool((a.isnan() == b.isnan()).all())
    a, b = a.nan_to_num(), b.nan_to_num()
    assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6).all()) and float((a != b).float().mean()) < 2e-2


@pytest.mark.parametrize("heads,kv,dim,vdim,rot", [(16, 4, 128, 128, 128), (3, 1, 64, 40, 64), (5, 5, 64, 64, 16), (2, 1, 256, 256, 0), (7, 7, 128, 8, 120)])
@pytest.mark.parametrize("normed,mixed", itertools.product([False, True], [False, True]))
def test_softmax_attention(heads, kv, dim, vdim, rot, normed, mixed):
    announce(f"attn prepare rows {heads} {kv} {dim} {vdim} {rot} {normed} {mixed}")
    g, T, lib = torch.Generator().manual_seed(heads * dim + rot), 259, _lib.load_decoder()
    cols = heads * dim + kv * (dim + vdim)
    p, first = values(g, T, cols), values(g, T, kv * vdim + 8)
    row = lib.ed_attn_row_elems(kv, dim, vdim)
    norms = [torch.rand(dim, generator=g).cuda() + 0.5 for _ in range(2)]
    freq, mix = (10000.0 ** -(torch.arange(max(rot // 2, 1)) / max(rot // 2, 1))).float().cuda(), torch.tensor(0.3).cuda()
    positions = torch.arange(T, dtype=torch.int32).cuda() * 37
    order = torch.randperm(T, generator=g).int().cuda()
    out = []
    for step in (T, FEW):
        q_rows, cache = (torch.full((T, n), float("nan"), dtype=BF16, device="cuda") for n in (heads * dim, row))
        for t in range(0, T, step):
            n = min(step, T - t)
            a = _lib.AttnArgs(q=p[t].data_ptr(), k=p[t].data_ptr() + 2 * heads * dim, v=p[t].data_ptr() + 2 * (heads + kv) * dim, stride=cols,
                              q_norm=norms[0].data_ptr() if normed else None, k_norm=norms[1].data_ptr() if normed else None,
                              inv_freq=freq.data_ptr(), positions=positions[t:].data_ptr(), cache_rows=order[t:].data_ptr(), cache=cache.data_ptr(),
                              q_rows=q_rows[t].data_ptr(), T=n, heads=heads, kv_heads=kv, dim=dim, vdim=vdim, rot=rot, dtype=_lib.DTYPE_BF16,
                              scale=1.0, eps=1e-6)
            if mixed:
                a.mix, a.v_first, a.v_first_stride = mix.data_ptr(), first[t].data_ptr(), first.stride(0)
            assert lib.ed_attn_prepare(a, _lib.current_stream(p.device)) == 0
        out.append((q_rows, cache))
    for got, want in zip(*out):
        assert not bool(want.isnan().any())
        same(got, want)


@pytest.mark.parametrize("heads,dim,rot,rank", [(16, 128, 64, 512), (3, 24, 16, 40), (5, 64, 0, 256), (1, 8, 128, 504)])
def test_latent_attention(heads, dim, rot, rank):
    announce(f"latent prepare rows {heads} {dim} {rot} {rank}")
    g, T, lib = torch.Generator().manual_seed(heads * dim + rank), 259, _lib.load_decoder()
    q_cols, cols = heads * (dim + rot), heads * (dim + rot) + rank + rot
    cols += -cols % 8
    base = values(g, T, cols)
    weight, freq = torch.rand(rank, generator=g).cuda() + 0.5, (10000.0 ** -(torch.arange(max(rot // 2, 1)) / max(rot // 2, 1))).float().cuda()
    positions, order = torch.arange(T, dtype=torch.int32).cuda() * 37, torch.randperm(T, generator=g).int().cuda()
    out = []
    for step in (T, FEW):
        p, cache = base.clone(), torch.full((T, lib.ed_latent_row_elems(rank, rot)), float("nan"), dtype=BF16, device="cuda")
        for t in range(0, T, step):
            a = _lib.LatentArgs(q=p[t].data_ptr(), q_stride=cols, down=p[t].data_ptr() + 2 * q_cols, down_stride=cols, latent_w=weight.data_ptr(),
                                inv_freq=freq.data_ptr(), positions=positions[t:].data_ptr(), cache_rows=order[t:].data_ptr(),
                                cache=cache.data_ptr(), T=min(step, T - t), heads=heads, dim=dim, rot=rot, rank=rank, dtype=_lib.DTYPE_BF16,
                                scale=1.0, eps=1e-6)
            assert lib.ed_latent_prepare(a, _lib.current_stream(p.device)) == 0
        out.append((p, cache))
    for got, want in zip(*out):
        assert not bool(want.isnan().any())
        same(got, want)
