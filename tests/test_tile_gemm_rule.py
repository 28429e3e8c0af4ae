"""Which products the tiled kernel takes, and what its entry point refuses (nothing runs on a GPU here)."""
import itertools

import pytest
import torch

from electrock_infer_amd import _lib
from electrock_infer_amd.layers import decoder_ops as ops

F32, BF16 = _lib.DTYPE_F32, _lib.DTYPE_BF16


def test_the_rule():
    lib = _lib.load_decoder()
    # long prompts are the library's; whole results of few rows in a decode batch, and short sums of one, another kernel's
    for T, N, K in itertools.product((0, 8192), (2048, 4096, 12288), (1024, 2048, 4096)):
        assert lib.ed_tile_gemm_splits(T, N, K) == 0, (T, N, K)
        assert not any(lib.ed_tile_gemm_pays(T, N, K, act) for act in (0, 1, 2)), (T, N, K)
    for T, K in itertools.product((1, 16, 40, 64), (64, 512, 2048, 12288)):
        assert not any(lib.ed_tile_gemm_pays(T, N, K, act) for N, act in ((4096, 0), (4096, 1), (2048, 2)))
        assert (lib.ed_tile_gemm_splits(T, 4096, K) > 0) == (K > 2048 or (K == 2048 and T > 16))
        assert lib.ed_tile_gemm_pays(T, 12288, K, 0) == 1 and lib.ed_tile_gemm_pays(T, 8192, max(K, 1024), 2) == 1
    assert [lib.ed_tile_gemm_pays(T, 8192, 1024, 0) for T in (32, 33)] == [lib.ed_tile_gemm_pays(T, 6144, 4096, 0) for T in (4, 5)] == \
        [lib.ed_tile_gemm_pays(T, 4096, 2048, 2) for T in (8, 9)] == [0, 1]
    assert lib.ed_tile_gemm_pays(300, 6144, 2048, 1) == lib.ed_tile_gemm_pays(1024, 4096, 2048, 2) == lib.ed_tile_gemm_pays(1344, 2048, 512, 0) == 1
    assert lib.ed_tile_gemm_pays(2048, 1344, 512, 0) == 1                      # (the sides' roles do not matter)
    assert lib.ed_tile_gemm_pays(300, 6144, 2048, 3) == lib.ed_tile_gemm_pays(300, 6144, 2050, 0) == lib.ed_tile_gemm_pays(300, 512, 512, 0) == 0
    # ranges of K never shorter than two steps, and a decode batch's widest shapes stay whole
    for T, N, K in itertools.product((65, 200, 512), (1024, 2048, 4096, 12288), (512, 576, 2048, 12288)):
        splits = lib.ed_tile_gemm_splits(T, N, K)
        assert 1 <= splits <= 8 and splits * 2 <= K // 64, (T, N, K)


@pytest.mark.parametrize("change,code", [({"T": -1}, -4), ({"K": 100}, -4), ({"N": 0}, -4), ({"splits": 0}, -2), ({"splits": 3, "K": 128}, -2),
                                         ({"splits": 2}, -2), ({"act": 3}, -2), ({"act": 1, "dtype": F32}, -2), ({"x_stride": 64}, -2),
                                         ({"w_stride": 64}, -2), ({"dtype": 7}, -3), ({"x": None}, -1), ({"w": 24}, -7), ({"out": 8}, -7),
                                         ({"x_stride": 132}, -7), ({"T": 1 << 21}, -4), ({"T": 1 << 20, "N": 1 << 21}, -4)])
def test_refused(change, code):
    a = {"x": 16, "x_stride": 128, "w": 16, "w_stride": 128, "out": 16, "dtype": BF16, "splits": 1, "T": 100, "N": 64, "K": 128, "act": 0, **change}
    assert _lib.load_decoder().ed_tile_gemm(a["x"], a["x_stride"], a["w"], a["w_stride"], a["out"], a["dtype"], a["splits"], a["T"], a["N"], a["K"],
                                            a["act"], None) == code


def test_no_rows_are_no_work():
    assert _lib.load_decoder().ed_tile_gemm(None, 64, None, 64, None, BF16, 1, 0, 64, 64, 0, None) == 0


def test_host_tensors_and_gradients_are_the_librarys():
    x, w = torch.randn(100, 512).to(torch.bfloat16), torch.randn(1024, 512).to(torch.bfloat16)
    assert not ops._tiles_fit(x, w) and torch.equal(ops.linear(x, w), torch.nn.functional.linear(x, w))
    assert ops._plain(x, w) and not ops._plain(x.requires_grad_(), w)


def test_partial_sums_are_the_tiled_kernels_or_whole(monkeypatch):
    # us as two ranges of the weight-streaming kernel / of the tiled one, with the norm behind them, 64 tokens: 6144 x 1024 16.6 / 12.8,
    # 8192 x 1024 18.5 / 14.6, 8192 x 2048 20.7 / 17.4
    lib, calls = _lib.load_decoder(), []
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda t: True), raising=False)
    monkeypatch.setattr(ops, "_tile_gemm", lambda x, w, out, splits, cols, act: calls.append(("tile", splits)) or out)
    monkeypatch.setattr(ops, "_decode_gemm", lambda x, w, out, splits, cols, act: calls.append(("stream", splits)) or out)
    for T, N, K, want in ((33, 6144, 1024, ("tile", 2)), (64, 6144, 1024, ("tile", 2)), (33, 8192, 1024, ("tile", 2)), (64, 8192, 1024, ("tile", 2)),
                          (33, 8192, 2048, ("tile", 2)), (64, 8192, 2048, ("tile", 2)), (64, 5632, 1024, ("tile", 2)), (64, 12288, 2048, ("tile", 1)),
                          (24, 8192, 2048, ("tile", 1)), (24, 6144, 1024, ("stream", 1)), (8, 2048, 2048, ("stream", lib.ed_decode_gemm_splits(8, 2048, 2048)))):
        x, w = torch.zeros(T, K, dtype=torch.bfloat16), torch.zeros(N, K, dtype=torch.bfloat16)
        for exact in (False, True):
            out = ops.linear_parts(x, w, exact)
            assert calls.pop() == want and not calls, (T, N, K)
            assert out.shape[-2:] == (T, N) and out.dtype == (torch.float32 if exact or out.dim() == 3 else torch.bfloat16)
        # 0 says that another product is the faster one, not that this one stays whole
        if lib.ed_tile_gemm_splits(T, N, K) == 1:
            assert lib.ed_decode_gemm_splits(T, N, K) == 1
    # wherever the rule takes partial sums, the other kernel is not asked
    for T, N, K in itertools.product((17, 33, 64), range(512, 16384, 512), (1024, 1088, 2048, 6144)):
        assert lib.ed_tile_gemm_splits(T, N, K) >= 1, (T, N, K)


def test_where_the_rule_ends():
    pays = _lib.load_decoder().ed_tile_gemm_pays
    # sections and widths of few rows: to so many tokens, by K; with an activation further
    for rows, K, to in ((128, 512, 8192), (512, 512, 8192), (1024, 512, 8192), (1536, 512, 2048), (128, 1024, 8192), (256, 1024, 4096), (512, 1024, 2048),
                        (1024, 1024, 2048), (72, 2048, 0), (512, 1536, 0), (1024, 2048, 0), (512, 4096, 0)):
        assert [pays(T, rows, K, 0) for T in (1536, 2048, 4096, 8192, 8193, 16384)] == [int(T <= to) for T in (1536, 2048, 4096, 8192, 8193, 16384)], (rows, K)
    assert [pays(T, 192, 2048, 0) for T in (2048, 3072, 4096, 4097)] == [0, 1, 1, 0]
    for rows, K, to in ((512, 512, 16384), (1024, 1024, 8192), (512, 2048, 2048), (1024, 2048, 8192), (512, 4096, 0)):
        assert [pays(T, rows, K, 1) for T in (2048, 8192, 16384, 16385)] == [int(T <= to) for T in (2048, 8192, 16384, 16385)], (rows, K)
        assert [pays(T, rows // 2, K, 2) for T in (2048, 8192, 16384, 16385)] == [pays(T, rows, K, 1) for T in (2048, 8192, 16384, 16385)]
    # more tokens than rows of a short prompt, on wide weights
    assert [pays(1344, N, 512, 0) for N in (2048, 3072)] == [pays(1152, N, 256, 0) for N in (2048, 4096)] == [1, 0]
    assert [pays(T, 8192, 1024, 0) for T in (256, 448, 640)] == [1, 1, 0] and [pays(T, 16384, 1024, 1) for T in (512, 640)] == [1, 0]
    assert [pays(100, N, K, 0) for N, K in ((2048, 2048), (4096, 4096), (8192, 4096), (4096, 2048))] == [1, 0, 1, 1]
    # results that are stored one by one
    assert [pays(2048, N, 512, 0) for N in (1001, 1301, 1300)] == [pays(100, 4098, 2048, 0), pays(300, 4098, 2048, 0), 1] == [1, 0, 1]
    # partial sums: within the tokens and rows that the estimate was fitted to
    splits = _lib.load_decoder().ed_tile_gemm_splits
    for T, N, K in itertools.product((1024, 1025, 2048, 16384), (72, 128, 512, 1020), (512, 2048, 8192)):
        assert splits(T, N, K) == 0, (T, N, K)
    assert splits(1025, 2048, 2048) == splits(300, 2050, 2048) == 0 < splits(1024, 2048, 2048) and splits(100, 2050, 2048) > 0
