"""Written-out latent attention: eight waves that share the tiles of the same queries agree with four, at the edges of their tiles."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


# sizes whose tiles, and whose results, are what the groups' LDS is sized by; sequences that end in their first tile, in an odd and in
# an even one
@pytest.mark.parametrize("dim,rot,vdim", [(24, 8, 16), (64, 0, 64), (32, 0, 128), (64, 32, 96), (128, 64, 128), (184, 72, 128)])
def test_eight_waves_like_four(dim, rot, vdim):
    announce(f"latent prompt waves {dim} {rot} {vdim}")
    H, D, lens, past = 16, dim + rot, [1, 64, 65, 127, 100], [0, 0, 64, 193, 612]
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
    four, eight = run(0), run(max(n + c for n, c in zip(lens, past)))
    for i, (n, c) in enumerate(zip(lens, past)):
        # the definition; weights rounded to bf16 (half a step is up to 2^-8 of a value), the result once more; float32 scores and exponentials
        qd, kd = q[qb[i]:qb[i] + n].double().view(n, H, D), k[kb[i]:kb[i] + n + c].double().view(-1, H, dim)
        if rot:
            kd = torch.cat((kd, kr[kb[i]:kb[i] + n + c, :rot].double().view(-1, 1, rot).expand(-1, H, -1)), 2)
        s = torch.stack([qd[:, h] @ kd[:, h].t() for h in range(H)]) * D ** -0.5
        s.masked_fill_(torch.arange(n + c, device=DEV)[None] > c + torch.arange(n, device=DEV)[:, None], float("-inf"))
        w = torch.softmax(torch.cat((s, sink.double().view(H, 1, 1).expand(-1, n, 1)), 2), 2)[..., :-1]
        v = vt[:, kb[i]:kb[i] + n + c].double().view(H, vdim, -1)
        want, size = (torch.stack([w[h] @ x[h].t() for h in range(H)], 1).view(n, -1) for x in (v, v.abs()))
        bound = size * (2.0 ** -8 + 4e-4) + want.abs() * 2.0 ** -8 + 1e-6
        for got in (four, eight):
            assert float(((got[qb[i]:qb[i] + n].double() - want).abs() / bound).max()) <= 1, i
