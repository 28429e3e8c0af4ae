"""The front of latent attention in one call against its two steps: sizes at which it is one launch and at which it is not, ragged ones, both types."""
from ctypes import byref

import pytest
import torch

from electrock_infer_amd import _lib
from electrock_infer_amd.layers.decoder_ops import head_gemm, pad_k

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 17, 63, 300])
@pytest.mark.parametrize("heads,dim,rot,rank", [(16, 128, 64, 512), (3, 20, 6, 50), (5, 8, 128, 9), (32, 64, 0, 256), (2, 300, 2, 64)])
def test_one_call_is_both_steps(dtype, T, heads, dim, rot, rank):
    lib, g = _lib.load_decoder(), torch.Generator().manual_seed(T * heads + dim)
    rand = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    stride = -(-(heads * (dim + rot) + rank + rot) // 8) * 8
    pitch, row = -(-rank // 8) * 8, lib.ed_latent_row_elems(rank, rot)
    p, uk = rand(T, stride), pad_k(rand(heads, rank, dim))
    w, freq = rand(rank).float(), torch.rand(max(rot // 2, 1), generator=g).cuda()
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    positions, rows = ints([3 * t for t in range(T)]), ints([T - 1 - t for t in range(T)])
    results = []
    for whole in (False, True):
        q, cache, q_lat = p.clone(), rand(1, 1).expand(T, row).contiguous() * 0 + 7, torch.full((T, heads, pitch), 5.0, dtype=dtype, device="cuda")
        a = _lib.LatentArgs(q=q.data_ptr(), q_stride=stride, down=q.data_ptr() + heads * (dim + rot) * q.element_size(), down_stride=stride,
                            latent_w=w.data_ptr(), inv_freq=freq.data_ptr(), positions=positions.data_ptr(), cache_rows=rows.data_ptr(),
                            cache=cache.data_ptr(), q_latent=q_lat.data_ptr(), T=T, n_seqs=T, max_q=1, table_width=1, block_size=T, splits=1,
                            heads=heads, dim=dim, rot=rot, rank=rank, dtype=_lib.dtype_code(dtype), scale=1.0, eps=1e-6)
        stream = _lib.current_stream(q.device)
        if whole:
            assert lib.ed_latent_front(byref(a), uk.data_ptr(), stream) == 0
        else:
            assert lib.ed_latent_prepare(byref(a), stream) == 0
            head_gemm(q, stride, dim + rot, uk, dim, q_lat, heads * pitch, pitch, T)
        results.append((q, cache, q_lat))
    (q, cache, q_lat), (q1, cache1, q_lat1) = results
    assert torch.equal(q_lat, q_lat1)
    # The latent's sum of squares runs in another order, and a turn's two products may be contracted otherwise: float32's last bits of the sum or
    # of either addend (of at most 6), which may turn a value's last bit.
    for one, other in ((q, q1), (cache, cache1)):
        assert ((one.float() - other.float()).abs() <= (torch.finfo(dtype).eps + 2.0 ** -20) * one.float().abs() + 6 * 2.0 ** -23).all()
    straight = torch.cat([torch.arange(dim) + h * (dim + rot) for h in range(heads)]).cuda()
    assert torch.equal(q[:, straight], p[:, straight]) and torch.equal(q1[:, straight], p[:, straight])
    assert torch.equal(cache[:, rank + rot:], cache1[:, rank + rot:]) and not cache[:, pitch + rot:].any()
