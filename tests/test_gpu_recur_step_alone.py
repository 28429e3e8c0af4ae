"""A decoding step of a recurrence: the same bits for a sequence alone and beside others, though few heads have wider workgroups."""
from ctypes import byref

import pytest
import torch

from electrock_infer_amd import _lib

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("delta", [False, True])
# small states, whose workgroups are the same; large ones in every form: rows that twice the threads do not share evenly, columns one by one, a
# state that takes twice the threads in any case
@pytest.mark.parametrize("H,G,dim,vdim,n", [(129, 3, 20, 12, 2), (130, 2, 48, 5, 2), (64, 8, 64, 64, 5), (8, 8, 32, 32, 40), (40, 8, 128, 128, 7), (64, 1, 128, 64, 5),
                                            (100, 4, 100, 72, 3), (100, 4, 96, 75, 3), (100, 4, 256, 64, 3), (90, 3, 80, 80, 3)])
def test_alone_and_beside_others(delta, H, G, dim, vdim, n):
    g = torch.Generator(device="cuda").manual_seed(H + dim + delta)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g) * 0.5
    ch = 2 * G * dim + H * vdim
    width = -(-(ch + H * vdim + 2 * H) // 8) * 8
    p, conv, bias, a_log, dt, skip, norm = rand(n, width).to(BF16), rand(ch, 4), rand(ch), rand(H), rand(H), rand(H), rand(vdim) + 1.0
    rings, states = rand(n, 4, ch).to(BF16), rand(n, H, dim, vdim)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")

    def step(rows):
        ring, state, out = rings.clone(), states.clone(), torch.empty(len(rows), H * vdim, dtype=BF16, device="cuda")
        x, slots, starts = p[rows].contiguous(), ints(rows), ints([3 * r for r in rows])
        at = lambda c: x.data_ptr() + 2 * c
        a = _lib.RecurArgs(q=at(0), k=at(G * dim), v=at(2 * G * dim), decay_in=at(ch + H * vdim), beta_in=at(ch + H * vdim + H) if delta else None,
                           gate=at(ch) if delta else None, stride=width, conv_w=conv.data_ptr(), conv_b=bias.data_ptr(), a_log=a_log.data_ptr(),
                           dt_bias=dt.data_ptr(), skip=None if delta else skip.data_ptr(), norm_w=norm.data_ptr() if delta else None,
                           ring=ring.data_ptr(), states=state.data_ptr(), out=out.data_ptr(), slots=slots.data_ptr(), starts=starts.data_ptr(),
                           n_seqs=len(rows), heads=H, kv_heads=G, dim=dim, vdim=vdim, taps=4, dtype=_lib.dtype_code(BF16), q_scale=dim ** -0.5,
                           unit_eps=1e-6 if delta else 0.0, eps=1e-6)
        assert _lib.load_decoder().ed_recur_step(byref(a), _lib.current_stream(x.device)) == 0
        return out, state

    assert H * n > 256 >= H
    out, state = step(list(range(n)))
    for r in range(n):
        one, state1 = step([r])
        assert torch.equal(one[0], out[r]) and torch.equal(state1[r], state[r])
