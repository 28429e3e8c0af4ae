"""One range of keys on eight waves: the rule ends where it was measured to pay, and leaves longer contexts to the rule that splits them."""
import pytest

from electrock_infer_amd import _lib

BF16 = _lib.DTYPE_BF16


def choices(kv_heads, dim, n, keys):
    lib = _lib.load_decoder()
    return lib.ed_attn_ranges(BF16, 4 * kv_heads, kv_heads, dim, dim, n, 1, keys), lib.ed_attn_splits(BF16, 4 * kv_heads, kv_heads, dim, dim, n, 1, keys)


@pytest.mark.parametrize("kv_heads,dim,n,keys", [(4, 128, 40, 2049), (4, 128, 43, 16384), (8, 64, 20, 8192), (4, 128, 64, 16385), (4, 128, 48, 100000), (4, 128, 32, 1537)])
def test_long_contexts_are_split(kv_heads, dim, n, keys):
    ranges, splits = choices(kv_heads, dim, n, keys)
    assert ranges == splits > 1


@pytest.mark.parametrize("kv_heads,dim,n,keys", [(4, 128, 40, 2048), (4, 128, 44, 4096), (4, 128, 48, 16384), (8, 64, 24, 8192), (4, 128, 64, 16384), (4, 128, 32, 1536)])
def test_a_range_to_a_workgroup(kv_heads, dim, n, keys):
    assert choices(kv_heads, dim, n, keys)[0] == 1
