"""Which calls put the token input's weights in operand order first, and that both ways agree at the edges of that rule."""
import pytest

from electrock_infer_amd import _lib


def pays(T, W, dim):
    return _lib.load_decoder().ed_token_side_pack_pays(T, W, dim) == 1


def test_lines():
    assert not any(pays(T, W, dim) for T in (256, 4096) for W, dim in ((128, 64), (128, 128), (256, 64), (256, 128), (384, 32), (768, 32)))
    assert all(pays(T, W, 64) for T in (1, 768, 8192) for W in (384, 1024, 2048, 4096))
    assert pays(4097, 256, 96) and not pays(4096, 256, 96) and pays(1, 256, 256) and not pays(8192, 128, 128)
    assert [pays(T, 384, 32) for T in (4096, 4097)] == [False, True] and pays(2048, 1024, 32) and not pays(2048, 896, 32)
    assert [pays(T, 1536, 32) for T in (4096, 4097, 8192, 8193)] == [True, False, False, True] and pays(4097, 2048, 32) and pays(8192, 4096, 32)


def test_sizes_that_cannot_be_packed_never_are():
    assert not any(pays(8192, W, dim) for W, dim in ((2050, 64), (2048, 48), (8192, 64), (0, 64), (2048, 0)))


@pytest.mark.gpu
@pytest.mark.parametrize("T,W,dim", [(4096, 256, 96), (4097, 256, 96), (4096, 384, 32), (4097, 384, 32), (4097, 1152, 32), (8193, 1152, 32)])
def test_both_sides_of_the_lines(T, W, dim):
    from tests.test_gpu_token_side_packed import test_packed_weights
    test_packed_weights(W, T, dim, False)
