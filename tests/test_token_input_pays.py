"""The rule that takes the token input's gate and projection to the two launches that share them out: it ends where it was measured to pay."""
import pytest

from electrock_infer_amd import _lib


def pays(T, W, dim):
    return _lib.load_decoder().ed_token_input_pays(T, W, dim) == 1


# one by one is faster: narrow streams, and wide gates of few tokens, whose sums every workgroup of the projection adds up anew
@pytest.mark.parametrize("T,W,dim", [(300, 512, 32), (1280, 512, 32), (1, 1024, 64), (23, 512, 64), (300, 1024, 64), (1280, 1024, 64), (1, 8192, 128), (23, 2048, 128),
                                     (300, 4096, 128), (1280, 1024, 128)])
def test_one_by_one(T, W, dim):
    assert _lib.load_decoder().ed_token_input_parts(T, W, dim) > 0 and not pays(T, W, dim)


@pytest.mark.parametrize("T,W,dim", [(1, 256, 32), (64, 1024, 32), (300, 1024, 32), (1, 2048, 64), (23, 1024, 64), (23, 4096, 64), (300, 2048, 64), (1000, 4096, 64),
                                     (2244, 2048, 64), (64, 4096, 128), (128, 4096, 128), (300, 8192, 128), (1280, 2048, 128)])
def test_shared_out(T, W, dim):
    assert pays(T, W, dim)


def test_sizes_that_are_not_taken():
    assert not any((pays(0, 2048, 64), pays(1, 2048, 48), pays(1, 2000, 64), pays(1000, 2048, 64), pays(1 << 40, 2048, 64)))
