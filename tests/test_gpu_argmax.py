"""The greedy token: first of equal values, NaN above all, rows of any length."""
import pytest
import torch

from electrock_infer_amd.layers.decoder_ops import argmax_rows
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,V", [(1, 1), (3, 5), (2, 1023), (64, 4096), (1, 32000), (5, 32767), (7, 32768 + 4), (2, 100003)])
def test_places(T, V):
    announce(f"argmax {T} {V}")
    g = torch.Generator().manual_seed(V)
    x = torch.randn(T, V, generator=g)
    rows = [x, x.round(), torch.full((T, V), -float("inf")), torch.zeros(T, V), -x.abs() - 1.0]
    late = x.clone()
    late[:, -1] = 9.0
    nan = x.clone()
    nan[:, V // 2] = float("nan")
    nan[:, V - 1] = float("nan")
    inf = x.clone()
    inf[:, V // 3:] = float("inf")
    for r in rows + [late, nan, inf]:
        want = [next((i for i, v in enumerate(row) if v != v), None) for row in r.tolist()]
        want = [w if w is not None else row.index(max(row)) for w, row in zip(want, r.tolist())]
        assert argmax_rows(r.cuda()).tolist() == want
    assert argmax_rows(x.cuda().t().contiguous().t()).tolist() == x.argmax(-1).tolist()      # rows that do not lie whole
