"""The greedy token of rows at the lengths where the workgroup, or the vectors that a thread asks for at once, change."""
import pytest
import torch

from electrock_infer_amd.layers.decoder_ops import argmax_rows
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,V", [(3, 4), (2, 256), (2, 260), (3, 4092), (3, 4096), (2, 4100), (2, 8192), (2, 8196), (2, 16384), (2, 16388), (256, 16388), (300, 508)])
def test_places(T, V):
    announce(f"argmax lengths {T} {V}")
    g = torch.Generator().manual_seed(T + V)
    x = torch.randn(T, V, generator=g)
    last, few, nan, low = x.clone(), x.round(), x.clone(), torch.full((T, V), -float("inf"))
    last[:, -1] = 9.0
    nan[:, V // 2] = nan[:, -1] = float("nan")
    for r in (x, last, few, nan, low):
        # the first place of the largest value, a NaN above all
        top = torch.where(r.isnan().any(1, keepdim=True), r.isnan(), r == r.nan_to_num(nan=-float("inf"), neginf=-float("inf"), posinf=float("inf")).amax(1, keepdim=True))
        assert torch.equal(argmax_rows(r.cuda()).cpu().long(), top.float().argmax(1))
