"""Paged softmax attention with one group of 16 query rows to a portion and with several: another way to the cached rows, the same
results, at the edge between them and against float64."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce
from tests.test_gpu_attn_prompt import reference

pytestmark = pytest.mark.gpu
DEV, BLOCK, H, G = "cuda", 16, 8, 2


def attend(q, cache, tables, lens, past, dim, vdim, splits, dtype):
    T, n, out = sum(lens), len(lens), torch.full((sum(lens), H, vdim), float("nan"), dtype=dtype, device=DEV)
    begin = torch.tensor([sum(lens[:i]) for i in range(n + 1)], dtype=torch.int32, device=DEV)
    starts, spare = torch.full((n,), past, dtype=torch.int32, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV)
    po, pm = torch.full((T * H * splits * vdim,), float("nan"), device=DEV), torch.full((T * H * splits * 2,), float("nan"), device=DEV)
    a = _lib.AttnArgs(q=q.data_ptr(), k=q.data_ptr(), v=q.data_ptr(), stride=H * dim, positions=spare.data_ptr(), cache_rows=spare.data_ptr(),
                      cache=cache.data_ptr(), q_rows=q.data_ptr(), out=out.data_ptr(), part_o=po.data_ptr(), part_ml=pm.data_ptr(),
                      q_begin=begin.data_ptr(), starts=starts.data_ptr(), tables=tables.data_ptr(), T=T, n_seqs=n, max_q=max(lens),
                      table_width=tables.shape[1], block_size=BLOCK, splits=splits, heads=H, kv_heads=G, dim=dim, vdim=vdim, rot=0, window=0,
                      dtype=_lib.dtype_code(dtype), scale=dim ** -0.5, softcap=0.0, eps=1e-6)
    assert _lib.load_decoder().ed_attn_paged(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    return out.cpu()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (72, 136), (192, 64), (256, 256)])
@pytest.mark.parametrize("past,splits", [(0, 1), (63, 1), (200, 3)])
def test_one_group_and_several(dim, vdim, past, splits, dtype):
    announce(f"attn row groups {dim} {vdim} past {past} splits {splits} {dtype}")
    g = torch.Generator().manual_seed(dim + past)
    lens = [4, 1, 3, 5, 17]                                     # four rows of queries a token and key head: 16, 4, 12, 20 and 68
    pages = -(-(past + max(lens)) // BLOCK)
    q = torch.randn(sum(lens), H, dim, generator=g).to(dtype)
    cache = torch.randn(len(lens) * pages, BLOCK, G * (dim + vdim), generator=g).to(dtype)
    tables = torch.randperm(len(lens) * pages, generator=g).view(len(lens), pages)
    gpu = [t.to(DEV) for t in (q, cache, tables.int())]
    every = attend(gpu[0], gpu[1], gpu[2], lens, past, dim, vdim, splits, dtype)
    few = attend(gpu[0], gpu[1], gpu[2], lens[:3], past, dim, vdim, splits, dtype)
    assert torch.equal(every[:8], few)
    at = 0
    for n, pages_of in zip(lens, tables):
        rows = cache[pages_of].view(-1, G * (dim + vdim))[:past + n].double()
        kv = torch.cat((rows[:, :G * dim].view(-1, G, dim), rows[:, G * dim:].view(-1, G, vdim)), 2)
        want, size = reference(q[at:at + n].double(), kv, past, dim ** -0.5, 0.0, 0, vdim)
        # weights and results in the compute type: half a step is 2^-8 of a value in bf16; float32 sums and exponentials
        step = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
        bound = size * (step + 4e-4 if step else 2e-5) + want.abs() * step + 1e-6
        assert float(((every[at:at + n].double() - want).abs() / bound).max()) <= 1
        at += n
