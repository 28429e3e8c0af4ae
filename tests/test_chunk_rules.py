"""How many tokens a workgroup of the recurrent mixers' prompt kernels takes, by the work of a step."""
import pytest
import torch

from electrock_infer_amd.harness import FeguvikConfig, NunivikConfig
from electrock_infer_amd.harness.decoder_model import DecoderModel
from electrock_infer_amd.harness.feguvik import FeguvikForCausalLM, LayerSpec
from electrock_infer_amd.harness.nunivik import MixerSpec, NunivikForCausalLM


def feguvik(heads):
    gla = LayerSpec("gla", {"heads": heads, "dim": 8, "vdim": 8, "tau": 16.0}, 0, 1)
    with torch.device("meta"):
        return FeguvikForCausalLM(FeguvikConfig(vocab_size=8, width=64, layers=[gla], norm_eps=1e-6))


def nunivik(width):
    with torch.device("meta"):
        return NunivikForCausalLM(NunivikConfig(vocab_size=8, width=width, layers=[MixerSpec("attention", {"heads": 1, "kv_heads": 1, "dim": 8, "vdim": 8, "scale": 1.0}, 8)],
                                                norm_eps=1e-6))


def test_a_model_answers_for_all_tokens_by_default():
    assert DecoderModel().chunk_for([1000, 3]) == 256


def test_many_short_prompts_are_not_cut():
    model = feguvik(32)
    assert model.chunk_for([128] * 8) == 128 and model.chunk_for([60] * 4) == 128 and model.chunk_for([1000]) == 64 and model.chunk_for([100]) == 32
    assert feguvik(8).chunk_for([128] * 8) == 32 and model.chunk_for([8192]) == 256 and model.chunk_for([700] * 12) == 256


@pytest.mark.parametrize("width", [64, 512, 1024, 2048])
def test_narrow_models_go_by_tokens(width):
    """As the width of 2048 does; wider ones have more work per token."""
    model = nunivik(width)
    assert [model.chunk_for([n]) for n in (1, 1023, 1024, 4095, 4096, 8191, 8192)] == [64, 64, 128, 128, 256, 256, 512]
    assert nunivik(4096).chunk_for([600] * 5) == 256 and nunivik(4096).chunk_for([4096]) == 512


def test_lengths_are_whole_blocks():
    for model in (feguvik(1), feguvik(16), feguvik(64), nunivik(96), nunivik(4096)):
        assert all(model.chunk_for([n] * k) % 16 == 0 for n in (1, 33, 500, 8192) for k in (1, 7, 64))
