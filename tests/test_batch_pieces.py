"""The batch's one buffer: portions that are written as arrays, short ones among them, and decode steps."""
import pytest
import torch

from electrock_infer_amd.harness import SamplingParams
from electrock_infer_amd.harness.batch import ARRAY_TOKENS, DecodePadding, make_ragged
from electrock_infer_amd.harness.sequence import Sequence


def sequences(portions, block):
    out = []
    for i, (past, n) in enumerate(portions):
        s = Sequence([(7 * i + 3 * t) % 1009 for t in range(past + n + i)], SamplingParams())
        s.block_table, s.state_slot = [(11 * i + 5 * b) % 997 for b in range(-(-len(s) // block))], 40 - i
        s.num_computed_tokens, s.num_scheduled_tokens = past, n
        out.append(s)
    return out


A = ARRAY_TOKENS


@pytest.mark.parametrize("block", [1, 16, 24])
@pytest.mark.parametrize("portions", [[(0, 1)], [(5, 1), (0, 1), (33, 1)], [(0, A - 1), (3, A), (0, 2), (50, 3 * A + 1), (9, 1)], [(0, A), (A, A)], [(70, 2), (0, 1)]])
def test_every_number_stands_where_its_view_says(portions, block):
    seqs = sequences(portions, block)
    b = make_ragged(seqs, block, 16, "cpu")
    at = [p for past, n in portions for p in range(past, past + n)]
    owner = [s for s, (_, n) in zip(seqs, portions) for _ in range(n)]
    assert b.tokens.tolist() == [s.token_ids[p] for s, p in zip(owner, at)] and b.positions.tolist() == at
    assert b.cache_rows.tolist() == [s.block_table[p // block] * block + p % block for s, p in zip(owner, at)]
    ends = [sum(n for _, n in portions[:i]) for i in range(len(portions) + 1)]
    assert b.q_begin.tolist() == ends and b.logit_rows.tolist() == [e - 1 for e in ends[1:]]
    assert b.starts.tolist() == [p for p, _ in portions] and b.k_lens.tolist() == [p + n for p, n in portions]
    assert b.state_slots.tolist() == [40 - i for i in range(len(portions))]
    assert b.chunks.tolist() == [[i, ends[i] + t, min(16, n - t), 0] for i, (_, n) in enumerate(portions) for t in range(0, n, 16)]
    assert b.seq_chunks.tolist() == [sum(-(-n // 16) for _, n in portions[:i]) for i in range(len(portions) + 1)]
    for row, s, (past, n) in zip(b.tables.tolist(), seqs, portions):
        used = -(-(past + n) // block)
        assert row == s.block_table[:used] + [0] * (b.table_width - used)
    assert all(getattr(b, name).data_ptr() % 16 == 0 for name in ("tokens", "positions", "cache_rows", "tables", "chunks", "logit_rows"))
    assert all(v.dtype == torch.int32 for v in vars(b).values() if isinstance(v, torch.Tensor))


def test_padded_steps_overwrite_the_buffer():
    pad = DecodePadding(4, 8, 90, 3)
    first, second = sequences([(5, 1), (30, 1)], 16), sequences([(0, 1), (17, 1), (40, 1)], 16)
    kept = make_ragged(first, 16, 16, "cpu", padding=pad)
    make_ragged(second, 16, 16, "cpu", padding=pad, into=kept)
    fresh = make_ragged(second, 16, 16, "cpu", padding=pad)
    assert torch.equal(kept.buffer, fresh.buffer)
    assert fresh.tokens.tolist()[3] == 0 and fresh.cache_rows.tolist()[3] == 90 * 16 and fresh.state_slots.tolist()[3] == 3


def test_every_row_is_wanted_of_single_tokens_only():
    def seq(n, start, slot):
        s = Sequence([1] * (start + n), SamplingParams(temperature=0.0, max_tokens=4))
        s.block_table, s.state_slot, s.num_computed_tokens, s.num_scheduled_tokens = [slot], slot, start, n
        return s
    one, two = seq(1, 3, 0), seq(2, 0, 1)
    assert make_ragged([one], 16, 64, "cpu").every_row and make_ragged([one, seq(1, 0, 1)], 16, 64, "cpu").every_row
    assert not make_ragged([one, two], 16, 64, "cpu").every_row and not make_ragged([one], 16, 64, "cpu", rows=[0]).every_row
    padded = make_ragged([one], 16, 64, "cpu", padding=DecodePadding(4, 8, 9, 9))
    assert padded.every_row and padded.logit_rows.tolist() == [0, 1, 2, 3]
