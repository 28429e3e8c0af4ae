"""The pitch that the tiled product reads rows at, over every form of a matrix: 0 where a row would not start at a 16-byte boundary."""
import pytest
import torch

from electrock_infer_amd.layers import decoder_ops as ops


@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("columns", [8, 16, 20])
@pytest.mark.parametrize("stride", [4, 8, 16, 20, 24, 32])
@pytest.mark.parametrize("step", [1, 2])
@pytest.mark.parametrize("offset", [0, 4, 8])
def test_pitch_is_of_whole_aligned_rows(rows, columns, stride, step, offset):
    t = torch.empty(512, dtype=torch.bfloat16)
    assert t.data_ptr() % 16 == 0
    t = t.as_strided((rows, columns), (stride, step), offset)
    pitch = stride if rows > 1 else columns
    whole = step == 1 and pitch >= columns and pitch % 8 == 0 and offset % 8 == 0
    assert ops._pitch(t, columns) == (pitch if whole else 0)
