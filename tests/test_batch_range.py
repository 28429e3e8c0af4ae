"""Numbers of a batch that do not fit its 32-bit buffer are refused, in portions of every length."""
import struct

import pytest

from electrock_infer_amd.harness import SamplingParams
from electrock_infer_amd.harness.batch import ARRAY_TOKENS, make_ragged
from electrock_infer_amd.harness.sequence import Sequence


@pytest.mark.parametrize("n", [1, 2, ARRAY_TOKENS - 1, ARRAY_TOKENS, 3 * ARRAY_TOKENS])
@pytest.mark.parametrize("what", ["block", "row", "token", "negative"])
def test_numbers_beyond_32_bits_are_refused(n, what):
    s = Sequence([5] * n, SamplingParams())
    s.block_table, s.state_slot, s.num_scheduled_tokens = list(range(-(-n // 16))), 0, n
    make_ragged([s], 16, 16, "cpu")
    if what == "token":
        s.token_ids[-1] = 1 << 31
    else:
        s.block_table[-1] = {"block": 1 << 31, "row": 1 << 27, "negative": -(1 << 40)}[what]      # row: the block fits, its rows do not
    with pytest.raises((OverflowError, RuntimeError, struct.error)):
        make_ragged([s], 16, 16, "cpu")


def test_the_last_row_that_fits():
    s = Sequence([5] * 80, SamplingParams())
    s.block_table, s.state_slot, s.num_scheduled_tokens = [0, 1, 2, 3, (1 << 27) - 1], 0, 80
    assert make_ragged([s], 16, 16, "cpu").cache_rows.tolist()[-1] == (1 << 31) - 1
