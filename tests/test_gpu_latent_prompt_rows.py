"""Written-out latent attention: its workgroups of 64 and of 128 queries agree, at the edges of their tiles."""
import ctypes

import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dim,rot,vdim", [(24, 8, 16), (64, 0, 64), (64, 32, 96), (128, 64, 128), (184, 72, 128)])
def test_rows_per_workgroup(dim, rot, vdim):
    H, D = 32, dim + rot
    lens, past = [1, 63, 64, 65, 127, 128, 129, 190, 255], [0, 64, 1, 100, 7, 0, 63, 5, 130]
    announce(f"latent prompt rows {dim} {rot} {vdim}")
    g = torch.Generator().manual_seed(dim)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().to(DEV)
    keys = [-(-(n + c) // 64) * 64 for n, c in zip(lens, past)]
    begin = lambda sizes: [sum(sizes[:i]) for i in range(len(sizes) + 1)]
    qb, kb, K = begin(lens), begin(keys), sum(keys)
    q, k, kr, vt = rand(sum(lens), H * D), rand(K, H * dim), rand(K, max(rot, 8)), rand(H * vdim, K)
    sink = torch.randn(H, generator=g).to(DEV)

    def run(seqs):
        """The sequences ``seqs`` as one call -> the results of all rows."""
        i0, i1 = seqs[0], seqs[-1] + 1
        ints = [torch.tensor(v, dtype=torch.int32, device=DEV) for v in (qb[i0:i1 + 1], past[i0:i1], kb[i0:i1])]
        out = torch.full((sum(lens), H * vdim), float("nan"), dtype=torch.bfloat16, device=DEV)
        a = _lib.LatentPromptArgs(q=q.data_ptr(), q_stride=q.stride(0), k=k.data_ptr(), k_stride=k.stride(0), k_rot=kr.data_ptr(),
                                  k_rot_stride=kr.stride(0), vt=vt.data_ptr(), v_stride=K, out=out.data_ptr(), sink=sink.data_ptr(),
                                  q_begin=ints[0].data_ptr(), starts=ints[1].data_ptr(), k_begin=ints[2].data_ptr(), n_seqs=i1 - i0,
                                  max_q=max(lens[i0:i1]), heads=H, dim=dim, rot=rot, vdim=vdim, scale=D ** -0.5)
        assert _lib.load_decoder().ed_latent_prompt(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out[qb[i0]:qb[i1]]

    assert -(-max(lens) // 128) * H * len(lens) >= 512 > -(-max(lens) // 128) * H     # 128 queries at once, 64 one by one
    together, alone = run(range(len(lens))), torch.cat([run(range(i, i + 1)) for i in range(len(lens))])
    # The same sums in the same order; a compiler may join a product and a sum in one form and not in the other, so the float32
    # results may differ in their last bits and their roundings be neighbours (2^-7 of a value).
    assert bool(((together.double() - alone.double()).abs() <= alone.double().abs() * 2.0 ** -7).all())
    assert float((together != alone).double().mean()) < 1e-4
    # and the definition, for the longest
    i, n, c = len(lens) - 1, lens[-1], past[-1]
    qd, kd = q[qb[i]:].double().view(n, H, D), k[kb[i]:kb[i] + n + c].double().view(-1, H, dim)
    if rot:
        kd = torch.cat((kd, kr[kb[i]:kb[i] + n + c, :rot].double().view(-1, 1, rot).expand(-1, H, -1)), 2)
    s = torch.stack([qd[:, h] @ kd[:, h].t() for h in range(H)]) * D ** -0.5
    s.masked_fill_(torch.arange(n + c, device=DEV)[None] > c + torch.arange(n, device=DEV)[:, None], float("-inf"))
    w = torch.softmax(torch.cat((s, sink.double().view(H, 1, 1).expand(-1, n, 1)), 2), 2)[..., :-1]
    v = vt[:, kb[i]:kb[i] + n + c].double().view(H, vdim, -1)
    want, size = (torch.stack([w[h] @ x[h].t() for h in range(H)], 1).view(n, -1) for x in (v, v.abs()))
    # weights rounded to bf16 (half a step is up to 2^-8 of a value), the result once more; float32 scores and exponentials
    bound = size * (2.0 ** -8 + 4e-4) + want.abs() * 2.0 ** -8 + 1e-6
    assert float(((alone[-n:].double() - want).abs() / bound).max()) <= 1
