"""The long-portion attention kernel alone, against a float64 reference: scores inside, across and beyond the range in which the
soft cap's tanh is a polynomial, and portions that end at, before and behind the edges of its tiles of rows and keys."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
BF16, DEV, BLOCK = torch.bfloat16, "cuda", 16


def reference(q, kv, first, scale, cap, window, vdim):
    """-> outputs and the weighted mean of |v| (what a rounding of the weights is relative to)."""
    G, d = kv.shape[1], q.shape[2]
    pos = first + torch.arange(q.shape[0])
    gap = pos[:, None] - torch.arange(kv.shape[0])[None]
    hide = (gap < 0) | (gap >= (window or kv.shape[0]))
    out = []
    for h in range(q.shape[1]):
        k, v = kv[:, h * G // q.shape[1], :d], kv[:, h * G // q.shape[1], d:]
        s = q[:, h] @ k.t() * scale
        s = cap * torch.tanh(s / cap) if cap else s
        w = torch.softmax(s.masked_fill(hide, float("-inf")), 1)
        out.append(torch.stack((w @ v, w @ v.abs())))
    return torch.stack(out, 2)


@pytest.mark.parametrize("dim,vdim", [(64, 64), (72, 128), (128, 96), (128, 128), (256, 128), (40, 8)])
@pytest.mark.parametrize("n,first,window", [(1, 0, 0), (64, 0, 0), (65, 63, 40), (129, 5, 0), (200, 100, 130)])
@pytest.mark.parametrize("cap,strength", [(30.0, 1.0), (30.0, 4.5), (40.0, 40.0), (1.0, 1.0), (60.0, 4.0), (0.0, 1.0)])
def test_scores_in_every_form_of_the_cap(dim, vdim, n, first, window, cap, strength):
    announce(f"attn prompt {dim} {vdim} n {n} first {first} window {window} cap {cap} x {strength}")
    g = torch.Generator().manual_seed(dim + n)
    H, G, total = 4, 2, first + n
    q = (torch.randn(n, H, dim, generator=g) * strength).to(BF16)
    kv = torch.randn(total, G, dim + vdim, generator=g).to(BF16)
    blocks = -(-total // BLOCK)
    order = torch.randperm(blocks + 2, generator=g)[:blocks]
    cache = torch.full((blocks + 2, BLOCK, G * (dim + vdim)), float("nan"), dtype=BF16)      # keys of all heads, then values
    flat = torch.cat((kv[..., :dim].reshape(total, -1), kv[..., dim:].reshape(total, -1)), 1)
    for b in range(blocks):
        rows = flat[b * BLOCK:(b + 1) * BLOCK]
        cache[order[b], :len(rows)] = rows
    gpu = [t.to(DEV) for t in (q, cache, order.int().view(1, -1), torch.tensor([0, n]).int(), torch.tensor([first]).int())]
    out = torch.full((n, H, vdim), float("nan"), dtype=BF16, device=DEV)
    spare = torch.zeros(n, dtype=torch.int64, device=DEV)
    a = _lib.AttnArgs(q=gpu[0].data_ptr(), k=gpu[0].data_ptr(), v=gpu[0].data_ptr(), stride=H * dim, positions=spare.data_ptr(),
                      cache_rows=spare.data_ptr(), cache=gpu[1].data_ptr(), q_rows=gpu[0].data_ptr(), out=out.data_ptr(),
                      q_begin=gpu[3].data_ptr(), starts=gpu[4].data_ptr(), tables=gpu[2].data_ptr(), T=n, n_seqs=1, max_q=n,
                      table_width=blocks, block_size=BLOCK, splits=1, heads=H, kv_heads=G, dim=dim, vdim=vdim, rot=0, window=window,
                      dtype=_lib.DTYPE_BF16, scale=dim ** -0.5, softcap=cap, eps=1e-6)
    assert _lib.load_decoder().ed_attn_prompt(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    want, size = reference(q.double(), kv.double(), first, dim ** -0.5, cap, window, vdim)
    # The weights are rounded to bf16 (8 bits: half a step is up to 2^-8 of a value), their sum is not; the result is rounded
    # once more.  Scores of up to 40 * 5 in float32 and their exponentials add some 1e-4 of relative error.
    bound = size * (2.0 ** -8 + 4e-4) + want.abs() * 2.0 ** -8 + 1e-6
    worst = ((out.cpu().double() - want).abs() / bound).max().item()
    assert worst <= 1, worst


@pytest.mark.parametrize("dim,vdim", [(64, 64), (40, 8)])
@pytest.mark.parametrize("cap,strength", [(30.0, 1.0), (30.0, 4.5), (60.0, 4.0), (0.0, 1.0)])
def test_both_numbers_of_workgroups_to_a_cu(dim, vdim, cap, strength):
    """Portions that alone make 64 workgroups and together 576, which is more than two to a CU: the same sums in the same order."""
    n, first, window, S, H, G = 200, 37, 90, 9, 32, 8
    total, pages = first + n, -(-(first + n) // BLOCK)
    g = torch.Generator(device=DEV).manual_seed(dim)
    q = (torch.randn(S * n, H, dim, generator=g, device=DEV) * strength).to(BF16)
    cache = torch.randn(S * pages, BLOCK, G * (dim + vdim), generator=g, device=DEV).to(BF16)
    tables = torch.randperm(S * pages, generator=g, device=DEV).int().view(S, pages)
    spare = torch.zeros(S * n, dtype=torch.int64, device=DEV)

    def attend(at, count):
        announce(f"attn prompt groups {dim} {vdim} cap {cap} x {strength} portions {at} + {count}")
        begin = (torch.arange(count + 1, device=DEV) * n).int()
        starts, out = torch.full((count,), first, device=DEV).int(), torch.full((count * n, H, vdim), float("nan"), dtype=BF16, device=DEV)
        mine, pages_of = q[at * n:(at + count) * n].contiguous(), tables[at:at + count].contiguous()
        a = _lib.AttnArgs(q=mine.data_ptr(), k=mine.data_ptr(), v=mine.data_ptr(), stride=H * dim, positions=spare.data_ptr(), cache_rows=spare.data_ptr(),
                          cache=cache.data_ptr(), q_rows=mine.data_ptr(), out=out.data_ptr(), q_begin=begin.data_ptr(), starts=starts.data_ptr(),
                          tables=pages_of.data_ptr(), T=count * n, n_seqs=count, max_q=n, table_width=pages, block_size=BLOCK, splits=1, heads=H,
                          kv_heads=G, dim=dim, vdim=vdim, rot=0, window=window, dtype=_lib.DTYPE_BF16, scale=dim ** -0.5, softcap=cap, eps=1e-6)
        assert _lib.load_decoder().ed_attn_prompt(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out

    assert total <= pages * BLOCK
    together = attend(0, S)
    assert bool(torch.isfinite(together).all()) and torch.equal(together, torch.cat([attend(i, 1) for i in range(S)]))
