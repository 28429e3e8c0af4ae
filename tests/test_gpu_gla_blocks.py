"""Blocks of gated linear attention whose operands are loaded ahead (bf16, even sizes, up to eight waves): two blocks' operands lie
side by side and a block's norm ends in the next one.  Sizes with lanes, waves and channel tiles beyond the edges, chunks of one row up
to several blocks, and channels whose decay no factor can hold in some blocks.

The oracle in float64 on the same bf16 weights and rows; the bounds are those of the other bf16 cases of the mixer."""
import pytest
import torch

from tests.gpu_util import announce
from tests.test_gpu_decoder_ops import BF16, DEV, F, Feed, close, gla_module, rand

pytestmark = pytest.mark.gpu


# one wave with a channel tile more, ragged channels and columns, lanes beyond the block's rows, eight waves, two pairs per lane
@pytest.mark.parametrize("dim,vdim", [(2, 16), (30, 17), (20, 100), (50, 72), (62, 126), (64, 128), (100, 120), (128, 128)])
@pytest.mark.parametrize("far", [False, True])
def test_blocks_loaded_ahead(dim, vdim, far):
    announce(f"gla blocks {dim} x {vdim} far {far}")
    m, W, eps = {"heads": 2, "dim": dim, "vdim": vdim, "tau": 1.0 if far else 16.0}, 48, 1e-5
    mix, w = gla_module(W, m, 8, eps, BF16, spread=4.0 if far else 1.5)
    # (keys that are the queries: a first token's output is the sign of q.k times its value's norm, and bf16 rounds q.k)
    param, section = mix.TENSORS["k"]
    w["k"] = w["q"]
    mix.get_parameter(param).weight_loader(mix.get_parameter(param), w["k"].to(DEV), section)
    if far:                                            # e^-9 a token: beyond the limit in a whole block, within it in a short one
        w["a2.b"][::3] = -9.0
        mix.a2_bias.data.copy_(w["a2.b"])
    w = {"m." + k: t.double() for k, t in w.items()}
    hs = [rand(n, W, seed=70 + n).to(BF16).float() for n in (1, 16, 17, 31, 129)]
    want = [F.gated_linear_attention(h.double(), w, "m.", m, eps).float() for h in hs]
    for sizes in ([1000], [5, 16, 33]):
        states = torch.full((5, *mix.state_shape()), float("nan"), device=DEV)
        for got, ref in zip(Feed(hs, chunk=64).run(mix, states, sizes, BF16), want):
            close(got, ref, BF16, f32=5e-5)
