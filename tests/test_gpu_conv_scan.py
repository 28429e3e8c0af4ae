"""Recurrences of prompts: the convolution by few and by many tokens a wave, and the matrix scan of states for every width of its rows."""
import pytest
import torch

from electrock_infer_amd.harness import SamplingParams
from electrock_infer_amd.harness.batch import make_ragged
from electrock_infer_amd.harness.sequence import Sequence
from tests.gpu_util import DEV, announce
from tests.nunivik_util import delta, mamba
from tests.test_gpu_nunivik_ops import BF16, BLOCK, F32, recurrent, weights
from tests.test_gpu_recurrence_range import Case, close

pytestmark = pytest.mark.gpu


def call(mix, entry, p, lengths, starts):
    """Outputs, states and rings of one step of sequences of these lengths, behind `starts` tokens."""
    Sequence.block_size, seqs = BLOCK, []
    for i, (n, a) in enumerate(zip(lengths, starts)):
        s = Sequence([0] * (a + n), SamplingParams())
        s.block_table, s.state_slot, s.num_computed_tokens, s.num_scheduled_tokens = list(range(s.num_blocks)), i, a, n
        seqs.append(s)
    batch, cache = make_ragged(seqs, BLOCK, 64, DEV), mix.new_cache(0, BLOCK, len(lengths), DEV)
    g = torch.Generator().manual_seed(5)
    for t in (cache.states, cache.ring):
        t.copy_(torch.randn(1, *t.shape[1:], generator=g).to(t.dtype).expand(t.shape))
    m = entry["mixer"]
    named = {"beta": "beta", "gate": "gate", "norm": mix.norm, "q_scale": m["dim"] ** -0.5, "unit_eps": 1e-6} if entry["type"] == "delta" else {"skip": mix.skip}
    return mix.recur(p, batch, cache, **named).clone(), cache.states, cache.ring


# heads of 32, 16 and 64 lanes of the convolution, counts that leave lanes empty
@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("entry", [delta(32, 16, 128, 128, 4), delta(64, 64, 64, 64, 3), mamba(64, 1, 128, 64, 4), mamba(48, 2, 200, 60, 2)],
                         ids=lambda e: e["type"] + "-" + "-".join(str(v) for v in e["mixer"].values()))
def test_convolution_of_many_tokens_a_wave_like_of_few(entry, dtype):
    """A long sequence takes the step to 16 tokens a wave, the others alone go by four: the same bits (one order of every sum)."""
    announce(f"convolution {entry['mixer']} {dtype}")
    mix = recurrent(entry, 64, dtype, weights(entry, 64, 1))
    lengths, starts = [2, 3, 4, 5, 18, 67, 8000], [0, 7, 2, 0, 9, 1, 0]
    p = torch.randn(sum(lengths), mix.in_proj.out_rows, generator=torch.Generator().manual_seed(2)).to(dtype).to(DEV)
    many, at = call(mix, entry, p, lengths, starts), 0
    for i, n in enumerate(lengths[:-1]):
        out, states, ring = call(mix, entry, p[at:at + n].contiguous(), [n], [starts[i]])
        assert torch.equal(out, many[0][at:at + n]) and torch.equal(ring[0], many[2][i]), (i, n)
        # (alone a sequence of one chunk has no scan: one sum more or less)
        torch.testing.assert_close(states[0], many[1][i], rtol=1e-5, atol=1e-5 * float(many[1][i].abs().max()))
        at += n


# rows of less than a 16-byte piece's swap, of one, two, three, four, seven and eight tiles, and of two registers' worth
@pytest.mark.parametrize("dim,vdim", [(8, 20), (16, 16), (20, 24), (32, 16), (48, 40), (64, 64), (100, 24), (112, 128), (128, 48), (144, 16)])
@pytest.mark.parametrize("start", [0, 5])
def test_states_of_many_chunks(dim, vdim, start):
    announce(f"matrix scan {dim} {vdim} {start}")
    case = Case(delta(2, 1, dim, vdim, 1), 150, start=start)
    (_, states), (_, want) = case.run(16), case.want()
    close(states, want)
