"""The prompt kernel of softmax attention: workgroups of 64 and of 128 queries, each against the definition."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce
from tests.test_gpu_attn_prompt import BF16, BLOCK, DEV, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,vdim", [(64, 64), (96, 64), (72, 128), (128, 128), (256, 40)])
@pytest.mark.parametrize("cap,strength", [(30.0, 4.5), (60.0, 1.0), (0.0, 1.0)])
@pytest.mark.parametrize("window", [0, 90])
def test_both_sizes_of_workgroups(dim, vdim, cap, strength, window):
    """Portions that alone make 128 workgroups of 64 queries (or fewer) and together more than 512; the last one ends in a workgroup's
    first tile of queries."""
    lens, first, H, G = [200, 129, 64, 1, 255, 128, 100, 65], 37, 32, 8
    S, most = len(lens), max(lens)
    total, pages = first + most, -(-(first + most) // BLOCK)
    g = torch.Generator(device=DEV).manual_seed(dim)
    begin = [sum(lens[:i]) for i in range(S + 1)]
    q = (torch.randn(begin[-1], H, dim, generator=g, device=DEV) * strength).to(BF16)
    cache = torch.randn(S * pages, BLOCK, G * (dim + vdim), generator=g, device=DEV).to(BF16)
    tables = torch.randperm(S * pages, generator=g, device=DEV).int().view(S, pages)
    spare = torch.zeros(begin[-1], dtype=torch.int64, device=DEV)

    def attend(at, count):
        announce(f"attn prompt queries {dim} {vdim} cap {cap} x {strength} window {window} portions {at} + {count}")
        T = begin[at + count] - begin[at]
        qb, starts = torch.tensor([b - begin[at] for b in begin[at:at + count + 1]], device=DEV).int(), torch.full((count,), first, device=DEV).int()
        mine, pages_of = q[begin[at]:begin[at + count]].contiguous(), tables[at:at + count].contiguous()
        out = torch.full((T, H, vdim), float("nan"), dtype=BF16, device=DEV)
        a = _lib.AttnArgs(q=mine.data_ptr(), k=mine.data_ptr(), v=mine.data_ptr(), stride=H * dim, positions=spare.data_ptr(), cache_rows=spare.data_ptr(),
                          cache=cache.data_ptr(), q_rows=mine.data_ptr(), out=out.data_ptr(), q_begin=qb.data_ptr(), starts=starts.data_ptr(),
                          tables=pages_of.data_ptr(), T=T, n_seqs=count, max_q=max(lens[at:at + count]), table_width=pages, block_size=BLOCK, splits=1,
                          heads=H, kv_heads=G, dim=dim, vdim=vdim, rot=0, window=window, dtype=_lib.DTYPE_BF16, scale=dim ** -0.5, softcap=cap, eps=1e-6)
        assert _lib.load_decoder().ed_attn_prompt(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out.cpu().double()

    assert -(-most // 64) * H * S > 512 >= -(-most // 64) * H
    together = attend(0, S)
    flat = cache.cpu().double()
    for i in range(S):
        n = lens[i]
        rows = flat[tables[i].cpu().long()].reshape(-1, G * (dim + vdim))[:first + n]
        kv = torch.cat((rows[:, :G * dim].view(-1, G, dim), rows[:, G * dim:].view(-1, G, vdim)), 2)
        want, size = reference(q[begin[i]:begin[i + 1]].cpu().double(), kv, first, dim ** -0.5, cap, window, vdim)
        # weights rounded to bf16 (half a step is up to 2^-8 of a value), the result once more; float32 scores and exponentials some 1e-4
        bound = size * (2.0 ** -8 + 4e-4) + want.abs() * 2.0 ** -8 + 1e-6
        for got in (together[begin[i]:begin[i + 1]], attend(i, 1)):
            assert float(((got - want).abs() / bound).max()) <= 1, i
