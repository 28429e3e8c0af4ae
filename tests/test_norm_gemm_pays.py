"""The rule that takes a residual norm and the product behind it to one launch: it ends where it was measured to pay."""
import pytest

from electrock_infer_amd import _lib


def pays(T, N, K, act=0):
    return _lib.load_decoder().ed_norm_gemm_pays(T, N, K, act) == 1


# K whose steps do not come in fours, long gated rows, and the most rows of either number of tokens
@pytest.mark.parametrize("T,N,K,act", [(1, 12288, 2560, 0), (1, 16384, 3072, 0), (2, 9216, 3072, 0), (2, 12288, 3072, 1), (1, 6144, 4096, 2), (1, 8192, 4096, 2),
                                       (2, 6144, 4096, 2), (1, 8192, 3072, 2), (1, 12288, 1024, 0), (2, 8832, 2048, 0), (2, 12800, 4096, 0)])
def test_two_launches(T, N, K, act):
    assert _lib.load_decoder().ed_norm_gemm_supported(T, N, K, act) == 1 and not pays(T, N, K, act)


@pytest.mark.parametrize("T,N,K,act", [(1, 3072, 512, 0), (1, 8832, 2048, 0), (1, 4096, 2048, 2), (1, 8192, 2560, 0), (1, 12288, 3584, 0), (1, 16384, 4096, 0),
                                       (1, 4096, 4096, 2), (2, 8192, 2048, 1), (2, 12288, 4096, 0), (2, 4096, 4096, 2)])
def test_one_launch(T, N, K, act):
    assert pays(T, N, K, act)


def test_sizes_that_are_not_taken():
    assert not pays(3, 3072, 2048) and not pays(1, 3072, 2000) and not pays(1, 16400, 2048) and not pays(1, 3072, 4608) and not pays(0, 3072, 2048)
