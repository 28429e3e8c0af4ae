"""The prompt kernel of softmax attention under a soft cap: a portion's results are the same to the bit whether its workgroups have 64
queries, alone, or 128, beside other portions, though the two look at different scores together."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce
from tests.test_gpu_attn_prompt import BF16, BLOCK, DEV

pytestmark = pytest.mark.gpu


# scores inside, on both sides of and beyond the range of the cap's polynomial; portions that end in every 16 queries of a workgroup of 128
@pytest.mark.parametrize("dim,vdim", [(40, 8), (64, 64), (64, 128), (96, 64), (72, 128), (128, 128), (256, 40)])
@pytest.mark.parametrize("cap,strength", [(30.0, 1.0), (30.0, 4.5), (30.0, 40.0), (60.0, 4.0), (0.0, 1.0)])
@pytest.mark.parametrize("window", [0, 90])
def test_portions_alone_and_together(dim, vdim, cap, strength, window):
    lens, first, H, G = [200, 129, 64, 1, 255, 128, 100, 65, 170], 37, 32, 8
    S, most = len(lens), max(lens)
    pages = -(-(first + most) // BLOCK)
    g = torch.Generator(device=DEV).manual_seed(dim)
    begin = [sum(lens[:i]) for i in range(S + 1)]
    # (queries of very different sizes side by side, so that neighbours take different forms of the cap)
    q = (torch.randn(begin[-1], H, dim, generator=g, device=DEV) * torch.rand(begin[-1], H, 1, generator=g, device=DEV) * 2 * strength).to(BF16)
    cache = torch.randn(S * pages, BLOCK, G * (dim + vdim), generator=g, device=DEV).to(BF16)
    tables = torch.randperm(S * pages, generator=g, device=DEV).int().view(S, pages)
    spare = torch.zeros(begin[-1], dtype=torch.int64, device=DEV)

    def attend(at, count):
        announce(f"attn prompt alone {dim} {vdim} cap {cap} x {strength} window {window} portions {at} + {count}")
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
        return out

    assert -(-most // 64) * H * S > 800 and -(-most // 64) * H <= 512
    together = attend(0, S)
    assert bool(torch.isfinite(together).all()) and torch.equal(together, torch.cat([attend(i, 1) for i in range(S)]))
