"""How many partial sums the token input's gate product may leave: every range has a step of its kernel, or the call is refused in front of
any launch."""
import pytest

from electrock_infer_amd import _lib


def refusal(T, W, dim, n_parts):
    """The code for operands that are null: a bad number of ranges is found before they are."""
    return _lib.load_decoder().ed_token_input(None, None, None, None, None, 4 * dim, 0, None, n_parts, None, T, W, dim, None)


@pytest.mark.parametrize("W", [64, 192, 2048, 8192])
@pytest.mark.parametrize("T", [1, 64, 65, 300, 1280])
def test_no_range_is_empty(T, W):
    most = W // 32 if T <= 64 else min(W // 64, 64)
    assert _lib.load_decoder().ed_token_input_parts(T, W, 64) <= most
    for n, code in ((-1, -2), (0, -2), (1, -1), (most, -1), (most + 1, -2), (W // 32 + 1, -2)):
        assert refusal(T, W, 64, n) == code, n
