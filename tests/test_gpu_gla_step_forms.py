"""One decoding step of linear attention over the forms its loads branch on: ranks in eights or not, rows that begin at 16 bytes or not, heads of
one and of several turns of rows; against float64."""
from ctypes import byref

import pytest
import torch

from electrock_infer_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank,a2_stride,shift", [(16, 16, 0), (8, 24, 0), (16, 17, 0), (16, 16, 1), (13, 16, 0), (1, 1, 0)])
@pytest.mark.parametrize("dim,vdim", [(8, 4), (64, 128), (128, 96), (200, 5)])
def test_step_in_every_form(dtype, rank, a2_stride, shift, dim, vdim):
    g = torch.Generator().manual_seed(rank * dim + vdim)
    H, n = 2, 3
    rand = lambda *s: torch.randn(*s, generator=g)
    q, k, v, gate, a1 = (rand(n, w).to(dtype) for w in (H * dim, H * dim, H * vdim, H * vdim, rank))
    a2, bias, norm, states = rand(H * dim, a2_stride).to(dtype), rand(H * dim), rand(vdim) + 1.0, rand(n + 1, H, dim, vdim)
    starts, slots, tau = [5, 0, 9], [3, 0, 1], 4.0
    sizes = [0]
    for part in (q, k, v, gate):
        sizes.append(-(-(sizes[-1] + part.shape[1]) // 8) * 8)
    stride = -(-(sizes[-1] + shift + rank) // 8) * 8
    p = torch.zeros(n, stride, dtype=dtype)
    for at, part in zip(sizes[:4] + [sizes[4] + shift], (q, k, v, gate, a1)):
        p[:, at:at + part.shape[1]] = part
    dp, da2, dbias, dnorm, dst = (t.cuda() for t in (p, a2, bias, norm, states))
    out = torch.empty(n, H * vdim, dtype=dtype, device="cuda")
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    dstarts, dslots, at = ints(starts), ints(slots), lambda c: dp.data_ptr() + c * dp.element_size()
    a = _lib.GlaArgs(q=at(sizes[0]), k=at(sizes[1]), v=at(sizes[2]), g=at(sizes[3]), a1=at(sizes[4] + shift), stride=stride, a2=da2.data_ptr(),
                     bias=dbias.data_ptr(), norm_w=dnorm.data_ptr(), out=out.data_ptr(), slots=dslots.data_ptr(), starts=dstarts.data_ptr(),
                     states=dst.data_ptr(), n_seqs=n, heads=H, dim=dim, vdim=vdim, rank=rank, a2_stride=a2_stride, dtype=_lib.dtype_code(dtype),
                     tau=tau, q_scale=dim ** -0.5, eps=1e-6)
    assert _lib.load_decoder().ed_gla_step(byref(a), _lib.current_stream(dp.device)) == 0
    want = states.double().clone()
    for s in range(n):
        z = a2[:, :rank].double() @ a1[s].double() + bias.double()
        alpha = torch.exp(torch.nn.functional.logsigmoid(z) / tau).view(H, dim, 1)
        old = want[slots[s]].clone() if starts[s] else torch.zeros(H, dim, vdim, dtype=torch.float64)
        new = alpha * old + k[s].double().view(H, dim, 1) * v[s].double().view(H, 1, vdim)
        want[slots[s]] = new
        # float32: a product and a sum of rank terms in the exponent, then two roundings of each addend
        scale = (alpha * old).abs() * (1 + rank) + (k[s].double().view(H, dim, 1) * v[s].double().view(H, 1, vdim)).abs()
        assert ((dst[slots[s]].cpu().double() - new).abs() <= 2.0 ** -21 * (scale + 1e-6)).all()
        o = (q[s].double().view(H, dim, 1) * dim ** -0.5 * new).sum(1)
        o = o / (o.square().mean(-1, keepdim=True) + 1e-6).sqrt() * norm.double()
        gs = gate[s].double().view(H, vdim)
        o = (o * gs * torch.sigmoid(gs)).flatten()
        # one rounding to the type; a sum of dim terms beside it, against the row's largest
        assert ((out[s].cpu().double() - o).abs() <= torch.finfo(dtype).eps * o.abs() + dim * 2.0 ** -22 * o.abs().max() + 1e-6).all()
    untouched = [i for i in range(n + 1) if i not in slots]
    assert torch.equal(dst.cpu()[untouched], states[untouched])
