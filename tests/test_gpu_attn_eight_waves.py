"""Paged softmax attention whose contexts are not split, on eight waves: uneven lengths around the edges of 32, 256 and 512 keys, windows, soft caps and
ragged heads, against float64; and one range is what the layer asks for where every workgroup has a CU."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce
from tests.test_gpu_attn_prompt import reference

pytestmark = pytest.mark.gpu
BLOCK, BF16 = 16, torch.bfloat16


@pytest.mark.parametrize("H,G,dim,vdim", [(8, 2, 128, 128), (16, 1, 64, 64), (4, 4, 72, 136), (2, 1, 128, 256)])
@pytest.mark.parametrize("window,softcap", [(0, 0.0), (70, 0.0), (0, 30.0)])
def test_lengths(H, G, dim, vdim, window, softcap):
    announce(f"attn eight waves {H} {G} {dim} {vdim} {window} {softcap}")
    g = torch.Generator().manual_seed(dim + vdim + window)
    past = [0, 1, 30, 31, 32, 127, 128, 255, 256, 257, 511, 700, 5]
    n, pages = len(past), 64
    q = torch.randn(n, H, dim, generator=g).to(BF16)
    cache = torch.randn(n * pages, BLOCK, G * (dim + vdim), generator=g).to(BF16)
    tables = torch.randperm(n * pages, generator=g).view(n, pages)
    dq, dc, dt = q.cuda(), cache.cuda(), tables.int().cuda()
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    begin, starts, out = ints(list(range(n + 1))), ints(past), torch.full((n, H, vdim), float("nan"), dtype=BF16, device="cuda")
    a = _lib.AttnArgs(q=dq.data_ptr(), k=dq.data_ptr(), v=dq.data_ptr(), stride=H * dim, positions=begin.data_ptr(), cache_rows=begin.data_ptr(),
                      cache=dc.data_ptr(), q_rows=dq.data_ptr(), out=out.data_ptr(), q_begin=begin.data_ptr(), starts=starts.data_ptr(),
                      tables=dt.data_ptr(), T=n, n_seqs=n, max_q=1, table_width=pages, block_size=BLOCK, splits=1, heads=H, kv_heads=G, dim=dim,
                      vdim=vdim, rot=0, window=window, dtype=_lib.dtype_code(BF16), scale=dim ** -0.5, softcap=softcap, eps=1e-6)
    assert _lib.load_decoder().ed_attn_paged(ctypes.byref(a), _lib.current_stream(dq.device)) == 0
    for s in range(n):
        rows = cache[tables[s]].view(-1, G * (dim + vdim))[:past[s] + 1].double()
        kv = torch.cat((rows[:, :G * dim].view(-1, G, dim), rows[:, G * dim:].view(-1, G, vdim)), 2)
        want, size = reference(q[s:s + 1].double(), kv, past[s], dim ** -0.5, softcap, window, vdim)
        # weights and results in bf16: half a step is 2^-8 of a value; float32 sums and exponentials
        bound = size * (2.0 ** -8 + 4e-4) + want.abs() * 2.0 ** -8 + 1e-6
        assert float(((out[s:s + 1].cpu().double() - want).abs() / bound).max()) <= 1


def test_one_range_where_every_workgroup_has_a_cu():
    ranges, splits = _lib.load_decoder().ed_attn_ranges, _lib.load_decoder().ed_attn_splits
    for dtype, dim, n, q, keys in ((1, 128, 64, 1, 8192), (1, 128, 40, 4, 2048), (1, 64, 28, 1, 1536)):
        assert ranges(dtype, 16, 4, dim, 128, n, q, keys) == 1
    for dtype, dim, n, q, keys in ((1, 128, 65, 1, 8192), (1, 128, 28, 1, 1537), (1, 128, 39, 1, 4096), (1, 128, 40, 5, 2048), (1, 192, 64, 1, 8192), (0, 128, 64, 1, 2048)):
        assert ranges(dtype, 16, 4, dim, 128, n, q, keys) == splits(dtype, 16, 4, dim, 128, n, q, keys)
    assert ranges(1, 16, 3, 64, 64, 1, 1, 100) == 0 == ranges(1, 16, 4, 257, 64, 1, 1, 100) == ranges(1, 16, 4, 64, 64, 0, 1, 100)
