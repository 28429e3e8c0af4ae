"""The kernels of the token input by themselves, whatever the rule says: every number of ranges that is taken, at the edges of their tiles."""
import pytest
import torch

from electrock_infer_amd import _lib
from tests.gpu_util import announce
from tests.test_gpu_token_input import BF16, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 16, 17, 64, 65, 129, 512, 1281])
@pytest.mark.parametrize("W,dim", [(64, 32), (192, 64), (832, 128), (2112, 32)])
def test_every_number_of_ranges(T, W, dim):
    announce(f"token input kernels {T} {W} {dim}")
    g = torch.Generator(device="cuda").manual_seed(T * W + dim)
    rand = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device="cuda") * scale).to(BF16)
    x, gate, proj, table = rand(T, W), rand(dim, W, scale=W ** -0.5), rand(W, dim, scale=dim ** -0.5), rand(50, 3 * dim)
    tokens = torch.randint(0, 50, (T,), generator=g, device="cuda").int()
    lib = _lib.load_decoder()
    for n in {1, lib.ed_token_input_parts(T, W, dim), W // 32 if T <= 64 else min(W // 64, 64)}:
        sums, out = torch.full((n, T, dim), float("nan"), device="cuda"), torch.full((T, W), float("nan"), dtype=BF16, device="cuda")
        assert lib.ed_token_input(x.data_ptr(), gate.data_ptr(), proj.data_ptr(), tokens.data_ptr(), table.data_ptr(), table.stride(0), dim,
                                  sums.data_ptr(), n, out.data_ptr(), T, W, dim, _lib.current_stream(x.device)) == 0
        check(out, x, gate, proj, tokens, table, dim)
