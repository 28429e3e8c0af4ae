"""Written-out latent attention: a query's sums are the same to the bit whatever is known of the call's longest context."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


# every number of 32-element steps of a key, both numbers of value columns; portions that end in every 16 queries of a workgroup, their
# contexts in an odd and in an even tile; queries that see one key of a tile, and none
@pytest.mark.parametrize("dim,rot,vdim", [(24, 8, 16), (64, 0, 64), (40, 24, 128), (64, 32, 96), (96, 0, 64), (96, 32, 128), (128, 64, 64), (128, 64, 128), (184, 72, 128)])
def test_known_and_unknown_contexts(dim, rot, vdim):
    announce(f"latent prompt order {dim} {rot} {vdim}")
    H, D, lens, past = 16, dim + rot, [1, 64, 65, 127, 100, 17], [0, 0, 64, 193, 612, 383]
    g = torch.Generator().manual_seed(dim)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().to(DEV)
    keys = [-(-(n + c) // 64) * 64 for n, c in zip(lens, past)]
    begin = lambda sizes: [sum(sizes[:i]) for i in range(len(sizes) + 1)]
    qb, kb, K = begin(lens), begin(keys), sum(keys)
    q, k, kr, vt = rand(sum(lens), H * D), rand(K, H * dim), rand(K, max(rot, 8)), rand(H * vdim, K)
    sink = torch.randn(H, generator=g).to(DEV)
    ints = [torch.tensor(v, dtype=torch.int32, device=DEV) for v in (qb, past, kb[:-1])]

    def run(max_context):
        out = torch.full((sum(lens), H * vdim), float("nan"), dtype=torch.bfloat16, device=DEV)
        a = _lib.LatentPromptArgs(q=q.data_ptr(), q_stride=q.stride(0), k=k.data_ptr(), k_stride=k.stride(0), k_rot=kr.data_ptr(),
                                  k_rot_stride=kr.stride(0), vt=vt.data_ptr(), v_stride=K, out=out.data_ptr(), sink=sink.data_ptr(),
                                  q_begin=ints[0].data_ptr(), starts=ints[1].data_ptr(), k_begin=ints[2].data_ptr(), n_seqs=len(lens),
                                  max_q=max(lens), heads=H, dim=dim, rot=rot, vdim=vdim, scale=D ** -0.5)
        assert _lib.load_decoder().ed_latent_prompt_behind(ctypes.byref(a), max_context, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out

    assert -(-max(lens) // 64) * H * len(lens) <= 384
    unknown = run(0)
    assert bool(torch.isfinite(unknown).all()) and torch.equal(unknown, run(max(n + c for n, c in zip(lens, past))))
