"""A per-layer token input whose weights are written after loading was finished: prompts read what is there now, as short portions do."""
import pytest
import torch

from electrock_infer_amd.layers.token_side import TokenSideInput
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
W, DIM, T = 1024, 64, 70


def close(side, one_launch, inputs):
    x, y, post, tokens, table, nxt = inputs
    side.ONE_LAUNCH_ROWS = 0 if one_launch else 10 ** 9
    stream, out = x.clone(), torch.empty(T, W, dtype=torch.bfloat16, device="cuda")
    side.close_layer(stream, y, post, tokens, table, 1e-6, out, nxt)
    return stream


@pytest.mark.parametrize("how", ["data", "copy", "state_dict", "replace"])
def test_weights_written_after_loading(how):
    announce(f"token side, weights written by {how}")
    g = torch.Generator().manual_seed(3)
    rand = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).cuda()
    side = TokenSideInput(W, DIM, 8, torch.bfloat16).cuda()
    weights = [{"gate": rand(DIM, W, scale=W ** -0.5).bfloat16(), "proj": rand(W, DIM, scale=DIM ** -0.5).bfloat16()} for _ in range(2)]
    inputs = (rand(T, W), rand(T, W).bfloat16(), 1 + rand(W, scale=0.2), torch.randint(0, 50, (T,), generator=g).int().cuda(),
              rand(50, DIM + 16).bfloat16(), 1 + rand(W, scale=0.2))

    def write(values):
        for name, v in values.items():
            if how == "data":
                getattr(side, name).data.copy_(v)
            elif how == "copy":
                getattr(side, name).copy_(v)
            elif how == "replace":
                setattr(side, name, torch.nn.Parameter(v.clone(), requires_grad=False))
        if how == "state_dict":
            side.load_state_dict({**side.state_dict(), **values})

    write(weights[0])
    side.finish_loading()
    first = close(side, True, inputs)
    for now in (weights[1], weights[0]):
        write(now)
        stream = close(side, True, inputs)
        assert torch.equal(stream, first) == (now is weights[0])
        # the same in steps: products, gates and sums rounded to bf16 at other places, 2^-8 of values of a few units each
        assert float((stream - close(side, False, inputs)).abs().max()) < 0.06
