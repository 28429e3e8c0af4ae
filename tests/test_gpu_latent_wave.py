"""Latent attention over the pages, bf16: the kernel whose waves work alone, at the edges of its row sizes, of its tiles of 16
keys, of the ranges of keys, and with scores that keep growing along the keys."""
import pytest
import torch

from tests.gpu_util import announce
from tests.test_gpu_decoder_ops import BF16, BLOCK, DEV, Feed, close, latent_oracle, mla, mla_module, rand

pytestmark = pytest.mark.gpu


def run(mix, h, sizes):
    feed = Feed([h])
    cache = torch.full((feed.num_blocks, BLOCK, mix.row_elems()), float("nan"), dtype=BF16, device=DEV)
    return feed.run(mix, cache, sizes, BF16)[0]


# rank, rotation: each form's largest row, the first that it no longer takes, ranks that are no multiple of a tile
@pytest.mark.parametrize("rank,rot", [(128, 64), (128, 72), (129, 2), (256, 64), (256, 66), (300, 12), (512, 64), (505, 64), (512, 66)])
def test_row_sizes(rank, rot):
    announce(f"latent wave {rank} {rot}")
    m = mla(17, 16, rot, 16, rank)
    mix, w = mla_module(64, m, 1e-5, BF16)
    h = rand(100, 64, seed=rank).to(BF16).float()
    want = latent_oracle(h, w, m, 1e-5)
    for sizes in ([33], [63, 1, 20, 1], [16, 1]):
        close(run(mix, h, sizes), want, BF16, bf16=3e-2)


@pytest.mark.parametrize("n", [15, 16, 17, 64, 65, 200])
@pytest.mark.parametrize("splits", [1, 2, 3, 7, 64])
def test_ranges_of_keys(n, splits, monkeypatch):
    """The last token against n keys, some ranges of them without a key, weights beyond e^8 from tile to tile."""
    announce(f"latent wave ranges {n} {splits}")
    m = mla(16, 16, 8, 16, 64, scale=1.5)
    mix, w = mla_module(64, m, 1e-5, BF16, q_scale=3.0)
    monkeypatch.setattr(mix, "splits", lambda batch: splits)
    h = rand(n, 64, seed=n)
    h[:, :8] += torch.linspace(0.0, 3.0, n)[:, None] * h[-1, :8].sign()      # the later, the more alike the last one
    h = h.to(BF16).float()
    want = latent_oracle(h, w, m, 1e-5)
    # (scores of a few dozen, from operands rounded to bf16: weights are off by a few per cent)
    close(run(mix, h, [n - 1, 1] if n < 64 else [40] * (n // 40) + [1] * (n % 40))[-1:], want[-1:], BF16, bf16=4e-2)
