"""Latent attention over the pages: how the keys are shared out, which kernel takes a call, and that both take every batch."""
import itertools

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce

F32, BF16 = _lib.DTYPE_F32, _lib.DTYPE_BF16


def plan(dtype, heads, rank, rot, n_seqs, max_q, keys):
    lib = _lib.load_decoder()
    return lib.ed_latent_waves(dtype, heads, rank, rot, n_seqs, max_q, keys), lib.ed_latent_splits(dtype, heads, rank, rot, n_seqs, max_q, keys)


def test_numbers_of_ranges():
    for dtype, heads, (rank, rot), n, q, keys in itertools.product((F32, BF16), (1, 16, 128), ((9, 2), (128, 64), (128, 128), (256, 128), (512, 64), (512, 128)),
                                                                   (1, 5, 64, 700), (1, 7, 63, 8192), (1, 128, 129, 1000, 100000)):
        waves, splits = plan(dtype, heads, rank, rot, n, q, keys)
        assert 1 <= splits <= min(64, -(-keys // 128))
        assert not waves or (dtype == BF16 and rank + rot <= 576)
    for bad in ((7, 16, 64, 32, 1, 1, 100), (BF16, 0, 64, 32, 1, 1, 100), (BF16, 16, 513, 32, 1, 1, 100), (BF16, 16, 64, 33, 1, 1, 100), (BF16, 16, 64, 32, 0, 1, 100),
                (BF16, 16, 64, 32, 1, 0, 100), (BF16, 16, 64, 32, 1, 1, 0)):
        assert plan(*bad) == (0, 0)


@pytest.mark.parametrize("rank,rot", [(128, 64), (128, 128), (256, 64), (512, 64)])
def test_decode_steps_work_alone_and_fill_the_chip_once(rank, rot):
    for n, heads, keys in ((1, 16, 1000), (8, 16, 1000), (23, 32, 1500), (64, 16, 3000), (64, 64, 1000), (32, 128, 1000)):
        waves, splits = plan(BF16, heads, rank, rot, n, 1, keys)
        assert waves and splits * n * -(-heads // 16) <= 256


def test_a_grid_that_32_bits_do_not_count_goes_to_the_other_kernel():
    """Decode sequences beside a long portion: workgroups for the longest one's rows, times sequences, of 256 threads each."""
    for rank, rot in ((128, 64), (512, 64)):
        assert plan(BF16, 64, rank, rot, 2000, 4096, 8000)[0] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("rank,rot", [(64, 32), (128, 128), (256, 64), (256, 128), (512, 64)])
@pytest.mark.parametrize("n_seqs,tokens,heads", [(1, 63, 16), (1, 50, 48), (3, 20, 16), (9, 63, 16), (5, 40, 32), (1, 9, 16), (8, 1, 128)])
def test_portions_of_many_rows(n_seqs, tokens, heads, rank, rot):
    """Row groups that fill part of a round of XCDs, whole rounds and several, in both kernels, against float64."""
    import ctypes
    past, block = 70, 16
    announce(f"latent rows {n_seqs} x {tokens} tokens, {heads} heads on {rank} + {rot}")
    g, dev = torch.Generator().manual_seed(rank + tokens), "cuda"
    lens = [max(1, tokens - 7 * i) for i in range(n_seqs)]
    T, pages = sum(lens), -(-(past + tokens) // block)
    cache = torch.randn(n_seqs * pages, block, rank + rot, generator=g).bfloat16()
    tables = torch.randperm(n_seqs * pages, generator=g).view(n_seqs, pages)
    q, ql = torch.randn(T, heads * (16 + rot), generator=g).bfloat16(), torch.randn(T, heads, rank, generator=g).bfloat16()
    sink, scale = torch.randn(heads, generator=g), (rank + rot) ** -0.5
    begin = [sum(lens[:i]) for i in range(n_seqs + 1)]
    seen = set()
    want, size = torch.empty(T, heads, rank, dtype=torch.float64), torch.empty(T, heads, rank, dtype=torch.float64)
    for i, n in enumerate(lens):
        rows = cache[tables[i]].view(-1, rank + rot)[:past + n].double()
        full = torch.cat((ql[begin[i]:begin[i + 1]].double(), q[begin[i]:begin[i + 1]].double().view(n, heads, 16 + rot)[..., 16:]), 2)
        s = torch.stack([full[:, h] @ rows.t() for h in range(heads)]) * scale
        s.masked_fill_(torch.arange(past + n)[None] > past + torch.arange(n)[:, None], float("-inf"))
        w = torch.softmax(torch.cat((s, sink.double().view(heads, 1, 1).expand(-1, n, 1)), 2), 2)[..., :-1]
        for out, v in ((want, rows[:, :rank]), (size, rows[:, :rank].abs())):
            out[begin[i]:begin[i + 1]] = torch.stack([w[h] @ v for h in range(heads)], 1)
    d = [t.to(dev) for t in (cache, tables.int(), q, ql, sink, torch.tensor(begin).int(), torch.full((n_seqs,), past).int())]
    spare = torch.zeros(max(T, 64), dtype=torch.int32, device=dev)
    waves, chosen = plan(BF16, heads, rank, rot, n_seqs, tokens, pages * block)
    for splits in {chosen, 1, 3}:
        out = torch.full((T, heads, rank), float("nan"), dtype=torch.bfloat16, device=dev)
        po, pm = torch.full((T * heads * splits * rank,), float("nan"), device=dev), torch.full((T * heads * splits * 2,), float("nan"), device=dev)
        a = _lib.LatentArgs(q=d[2].data_ptr(), q_stride=heads * (16 + rot), down=d[2].data_ptr(), down_stride=heads * (16 + rot), latent_w=spare.data_ptr(),
                            inv_freq=spare.data_ptr(), positions=spare.data_ptr(), cache_rows=spare.data_ptr(), cache=d[0].data_ptr(), q_latent=d[3].data_ptr(),
                            out=out.data_ptr(), sink=d[4].data_ptr(), q_begin=d[5].data_ptr(), starts=d[6].data_ptr(), tables=d[1].data_ptr(),
                            part_o=po.data_ptr(), part_ml=pm.data_ptr(), T=T, n_seqs=n_seqs, max_q=tokens, table_width=pages, block_size=block,
                            splits=splits, heads=heads, dim=16, rot=rot, rank=rank, dtype=BF16, scale=scale, eps=1e-6)
        assert _lib.load_decoder().ed_latent_paged(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        seen.add(splits)
        # weights rounded to bf16 (half a step is up to 2^-8 of a value), the result once more; float32 scores and exponentials
        bound = size * (2.0 ** -8 + 4e-4) + want.abs() * 2.0 ** -8 + 1e-6
        assert float(((out.double().cpu() - want).abs() / bound).max()) <= 1, (splits, waves)


def test_the_cases_above_reach_both_kernels_in_every_form():
    for rank, rot in ((128, 128), (256, 64), (256, 128), (512, 64)):
        routes = {plan(BF16, h, rank, rot, n, q, 144)[0] for n, q, h in ((1, 63, 16), (1, 50, 48), (3, 20, 16), (9, 63, 16), (5, 40, 32), (1, 9, 16), (8, 1, 128))}
        assert routes == {0, 1}, (rank, rot)
