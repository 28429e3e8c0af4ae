"""The end of a layer in one launch with its weights in operand order, against the same with the weights as they are."""
import pytest
import torch

from electrock_infer_amd import _lib
from electrock_infer_amd.layers.token_side import TokenSideInput
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu


# widths of every form (four, eight and sixteen pieces a lane), one and several turns of gate columns, rows behind whole groups
@pytest.mark.parametrize("W", [128, 1024, 1152, 2048, 2176, 4096])
@pytest.mark.parametrize("T,dim", [(1, 32), (9, 64), (513, 96), (530, 64)])
@pytest.mark.parametrize("last", [False, True])
def test_packed_weights(W, T, dim, last):
    announce(f"token side packed {W} {T} {dim} {last}")
    if not _lib.load_decoder().ed_token_side_supported(W, dim):
        pytest.skip("the rows and the partial products do not fit in LDS")
    g = torch.Generator().manual_seed(W + T)
    rand = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).cuda()
    side = TokenSideInput(W, dim, 8, torch.bfloat16).cuda()
    side.ONE_LAUNCH_ROWS = 0
    side.gate.data.copy_(rand(dim, W, scale=W ** -0.5))
    side.proj.data.copy_(rand(W, dim, scale=dim ** -0.5))
    side.norm.data.copy_(1 + rand(W, scale=0.2))
    x, y, post, nxt = rand(T, W), rand(T, W).bfloat16(), 1 + rand(W, scale=0.2), None if last else 1 + rand(W, scale=0.2)
    tokens, table = torch.randint(0, 50, (T,), generator=g).int().cuda(), rand(50, dim + 16).bfloat16()
    got = []
    for packed in (False, True):
        if packed:
            side.finish_loading()
            assert side.gate_packed is not None and "gate_packed" not in side.state_dict()
        stream, out = x.clone(), torch.full((T, W + 4), 7.0, dtype=torch.bfloat16, device="cuda")
        side.close_layer(stream, y, post, tokens, table, 1e-6, out[:, :W], nxt)
        assert bool((out[:, W:] == 7).all())
        got.append((stream, out[:, :W].float()))
    # the same products in the same order: nothing but the order of the rows' registers differs
    assert float((got[0][0] - got[1][0]).abs().max()) <= 2 ** -20 * float(x.abs().max()) and torch.equal(got[0][1], got[1][1])


# eight pieces a lane on both sides of the LDS that two workgroups share, with whole and ragged groups of rows
@pytest.mark.parametrize("W,dim", [(1280, 192), (1280, 256), (1408, 96), (1408, 128), (1536, 96), (2048, 256)])
@pytest.mark.parametrize("T", [512, 513, 521, 544])
def test_rows_of_a_wave_by_lds(W, T, dim):
    test_packed_weights(W, T, dim, False)
