"""The recurrences' prompt kernels multiply by the state in parts: they stay at float32's distance from 64 bits."""
import pytest
import torch

from tests.gpu_util import announce
from tests.nunivik_util import delta, mamba
from tests.test_gpu_nunivik_ops import EPS, F32, N, Feed, rand, recurrent, slots, weights

pytestmark = pytest.mark.gpu


# one and two pieces of a key per thread, heads that share a workgroup (with waves left over), columns and rows that end inside a tile;
# heads of more than eight column tiles, whose output pass has a workgroup of its own kind (of 9, 10 and 16 waves)
@pytest.mark.parametrize("entry", [delta(4, 2, 128, 128, 4), delta(2, 2, 256, 64, 4), delta(2, 1, 70, 40, 4), mamba(8, 1, 128, 64, 4, 2), mamba(6, 2, 40, 24, 4),
                                   mamba(2, 1, 200, 130, 4), delta(2, 1, 128, 256, 4), delta(2, 2, 40, 130, 4), delta(1, 1, 64, 160, 4), delta(1, 1, 256, 144, 4)],
                         ids=lambda e: e["type"] + "-" + "-".join(str(v) for v in e["mixer"].values()))
@pytest.mark.parametrize("a_log", [-12.0, 1.0])
def test_distance_from_64_bits(entry, a_log):
    announce(f"recurrence precision {entry} {a_log}")
    W, T, H = 256, 530, entry["mixer"]["heads"]
    w = weights(entry, W, 3)
    w["mix.A_log"], w["mix.dt_bias"] = torch.full((H,), a_log), torch.zeros(H)
    h = rand(T, W, seed=5)
    want = N.MIXERS[entry["type"]](h.double(), {k: t.double() for k, t in w.items()}, "mix.", entry["mixer"], EPS, {})
    for chunk, sizes in ((64, [T]), (512, [T]), (128, [201, T])):
        mix = recurrent(entry, W, F32, w)
        got = Feed([h], chunk=chunk).run(mix, slots(mix, 1), sizes, F32)[0].double().cpu()
        # a float32 rounding per token and state, and one per product of the two projections: 2^-24 sqrt(530 + 512) of a value
        assert float((got - want).norm() / want.norm()) < 2.0 ** -24 * (T + 2 * W) ** 0.5
