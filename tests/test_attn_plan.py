"""How the paged softmax attention shares its keys out."""
import itertools

from electrock_infer_amd import _lib
from electrock_infer_amd.layers.attention import SoftmaxAttention

F32, BF16 = _lib.DTYPE_F32, _lib.DTYPE_BF16


def test_numbers_of_ranges():
    splits = _lib.load_decoder().ed_attn_splits
    for dtype, (heads, kv), dim, n, q, keys in itertools.product((F32, BF16), ((1, 1), (16, 4), (64, 1)), (8, 128, 256), (1, 6, 64, 700), (1, 5, 47, 8192), (1, 128, 129, 1000, 100000)):
        s = splits(dtype, heads, kv, dim, 64, n, q, keys)
        steps = -(-keys // 128)
        assert 1 <= s <= min(64, steps)
        assert s == 1 or -(-steps // (s - 1)) > -(-steps // s)         # no range that leaves the longest as it is
    for bad in ((7, 16, 4, 64, 64, 1, 1, 100), (BF16, 16, 3, 64, 64, 1, 1, 100), (BF16, 16, 4, 257, 64, 1, 1, 100), (BF16, 16, 4, 64, 0, 1, 1, 100), (BF16, 16, 4, 64, 64, 0, 1, 100),
                (BF16, 16, 4, 64, 64, 1, 0, 100), (BF16, 16, 4, 64, 64, 1, 1, 0)):
        assert splits(*bad) == 0


def test_forms_that_wait_for_their_keys_have_more_workgroups_in_flight():
    """24 sequences of 2000 keys, 96 row groups: enough workgroups that others run while one waits (shares of 750 in flight)."""
    splits = lambda dtype, dim, vdim: _lib.load_decoder().ed_attn_splits(dtype, 16, 4, dim, vdim, 24, 1, 2000)
    assert 96 * splits(F32, 64, 64) >= 750 and 96 * splits(F32, 128, 128) >= 750 and 96 * splits(BF16, 64, 64) > 288 < 96 * splits(BF16, 192, 64)


def test_a_full_chip_is_split_behind_long_contexts_only():
    """64 sequences on four key heads: one row group for every CU."""
    splits = lambda n, keys: _lib.load_decoder().ed_attn_splits(BF16, 16, 4, 128, 128, n, 1, keys)
    assert [splits(64, k) for k in (128, 1024, 2048)] == [1, 1, 1] and splits(64, 4096) == 2 and splits(63, 2048) > 1


def test_a_window_bounds_the_keys():
    import torch
    batch = type("B", (), {"max_q": 1, "n_seqs": 1, "max_context": 8192})()
    make = lambda window: SoftmaxAttention(64, 16, 4, 64, 64, 1.0, 1e-6, torch.bfloat16, window=window)
    assert make(100).splits(batch) == 1 < make(1000).splits(batch) < make(0).splits(batch)
