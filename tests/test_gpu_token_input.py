"""The token input's gate and projection in two launches, against float64 and against the two one by one."""
import pytest
import torch

from electrock_infer_amd import _lib
from electrock_infer_amd.layers import decoder_ops as ops
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def check(got, x, gate, proj, tokens, table, column0):
    dim = gate.shape[0]
    want_g = torch.nn.functional.gelu(x.double() @ gate.double().t(), approximate="tanh") * table.double()[tokens.long(), column0:column0 + dim]
    want, size = want_g @ proj.double().t(), want_g.abs() @ proj.double().abs().t()
    # g rounded to bf16 (half a step is up to 2^-8 of a value), the result once more; float32 sums of at most 2112 products and the gelu 1e-4
    bound = size * (2.0 ** -8 + 1e-4) + want.abs() * 2.0 ** -8 + 1e-6
    assert bool(((got.double() - want).abs() <= bound).all())


# tokens at the edges of a workgroup's and of the tiled product's, and one below and above each rule; widths of one wave's columns, of
# ragged ranges and of several rounds of columns
@pytest.mark.parametrize("T", [1, 15, 16, 17, 64, 65, 128, 129, 512, 513, 1279, 1281])
@pytest.mark.parametrize("W,dim", [(64, 32), (192, 64), (832, 128), (2048, 64), (2112, 32)])
def test_gate_and_projection(T, W, dim):
    announce(f"token input {T} {W} {dim}")
    g = torch.Generator(device="cuda").manual_seed(T * W + dim)
    rand = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device="cuda") * scale).to(BF16)
    x, gate, proj, table = rand(T, W), rand(dim, W, scale=W ** -0.5), rand(W, dim, scale=dim ** -0.5), rand(50, 3 * dim)
    tokens = torch.randint(0, 50, (T,), generator=g, device="cuda").int()
    parts = _lib.load_decoder().ed_token_input_parts(T, W, dim)
    assert (parts == 0) == (512 < T < 1280 and W <= 2048) and parts <= max(1, W // 256)
    with torch.inference_mode():
        got = ops.token_input(x, gate, proj, tokens, table, dim)
    check(got, x, gate, proj, tokens, table, dim)


def test_one_by_one_where_operands_are_not_plain():
    announce("token input of other operands")
    x, gate, proj, table = (torch.randn(*s, device="cuda").to(BF16) for s in ((5, 128), (64, 128), (128, 64), (9, 66)))
    tokens = torch.arange(5, device="cuda").int()
    with torch.inference_mode():         # (rows of the table that no 8-byte load takes; float32)
        check(ops.token_input(x, gate, proj, tokens, table, 2), x, gate, proj, tokens, table, 2)
        check(ops.token_input(x.float(), gate.float(), proj.float(), tokens, table.float(), 2), x, gate, proj, tokens, table, 2)
