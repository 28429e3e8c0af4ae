"""Steps of one and two tokens whose residual norms go into the products behind them: whole models against the oracle, the rows themselves where
a product does not take them, and values that are no numbers."""
import pytest
import torch

from electrock_infer_amd import _lib
from electrock_infer_amd.harness.trace import TraceReplay
from electrock_infer_amd.layers import decoder_ops as ops
from tests import feguvik_util, nunivik_util
from tests.gpu_util import announce
from tests.test_gpu_feguvik import assert_close

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

# Widths that the product with a norm takes.  Feguvik: a loop over a layer without a feed-forward and one with, in front and behind it one each;
# Nunivik: every mixer, with a feed-forward and without
FEGUVIK = feguvik_util.config(512, 300, [(feguvik_util.mla(4, 64, 32, 64, 128), 384), (feguvik_util.gla(2, 64, 96, 8.0), None),
                                         (feguvik_util.mla(2, 48, 16, 40, 72), 200), (feguvik_util.gla(4, 64, 48, 16.0), 512)], side=32, loop=(1, 3, 2))
NUNIVIK = nunivik_util.config(512, 300, [(nunivik_util.attn(8, 2, 64, 64, cap=30.0, rot=64), 400), (nunivik_util.delta(4, 2, 64, 48, 3), None),
                                         (nunivik_util.mamba(4, 2, 48, 32, 4), 256), (nunivik_util.attn(4, 2, 48, 40, size=20, rot=32, mix=True), None),
                                         (nunivik_util.delta(2, 1, 32, 64, 4), 128)])
MODELS = {"feguvik": (feguvik_util, FEGUVIK, lambda: feguvik_util.random_weights(FEGUVIK, 16, 3)), "nunivik": (nunivik_util, NUNIVIK, lambda: nunivik_util.random_weights(NUNIVIK, 3))}


@pytest.mark.parametrize("name", sorted(MODELS))
def test_models_against_the_oracle(name, tmp_path, monkeypatch):
    announce(f"norms inside products: {name}")
    util, cfg, weights = MODELS[name]
    w = weights()
    path = feguvik_util.write_checkpoint(tmp_path / name, cfg, w)
    w = {k: v.float() for k, v in w.items()}
    toks = {k: feguvik_util.draw_tokens(cfg, 40, seed=s) for s, k in enumerate("ab")}
    want = {k: util.oracle_logits(t, w, cfg) for k, t in toks.items()}
    taken, product = [], ops.NormedRows.product
    monkeypatch.setattr(ops.NormedRows, "product", lambda self, *a: taken.append(product(self, *a)) or taken[-1])

    def run(counts):
        """Both requests: a first portion each, then one token at a time, alone and together."""
        replay, rows, at = TraceReplay.for_model(path, "bfloat16", 200), {k: [] for k in toks}, dict.fromkeys(toks, 0)
        for step in counts:
            out = replay.step([{"id": k, "tokens": toks[k][at[k]:at[k] + n], "want": list(range(n))} for k, n in step.items()], [])
            for (k, n), part in zip(step.items(), out.split(list(step.values()))):
                rows[k].append(part)
                at[k] += n
        return {k: torch.cat(v) for k, v in rows.items()}

    steps = [{"a": 5}, {"b": 3}] + [{"a": 1, "b": 1}] * 12 + [{"a": 1}] * 23 + [{"b": 1}] * 25
    got = run(steps)
    # products that read normed rows, seven a step: four of Feguvik's six layer runs have a feed-forward, and three go on to another run that opens
    # no pass of the loop; three of Nunivik's five layers have one, and four go on to another layer
    assert len(taken) == 60 * 7 and all(t is not None for t in taken)
    for k in toks:
        assert_close(got[k], want[k], "bfloat16", f"{name} {k}")
    # norms and products one by one: no closer to the oracle
    monkeypatch.setattr(ops.NormedRows, "product", lambda self, *a: None)
    apart = run(steps)
    for k in toks:
        one, two = feguvik_util.row_errors(got[k], want[k]).mean(), feguvik_util.row_errors(apart[k], want[k]).mean()
        assert float(one) < 1.25 * float(two), (float(one), float(two))


@pytest.mark.parametrize("gated", [False, True])
def test_rows_that_no_product_takes(gated):
    """More rows of weights than one launch pays for: the rows are made, the stream changes once and in place."""
    torch.manual_seed(1)
    T, K, rows = 2, 512, 8208
    assert _lib.load_decoder().ed_norm_gemm_supported(T, rows // 2 if gated else rows, K, 2 if gated else 0) == 1
    x, y, post = torch.randn(T, K, device="cuda"), torch.randn(3, T, K, device="cuda"), torch.rand(K, device="cuda") + 0.5
    w = (torch.randn(rows, K, device="cuda") * K ** -0.5).to(BF16)
    product = ops.linear_silu_gate if gated else ops.linear

    class Reader(torch.nn.Module):
        takes_normed_rows = True

        def forward(self, h):
            return product(h, w)

    reader, kept, want = Reader(), x.clone(), torch.empty(T, K, dtype=BF16, device="cuda")
    ops.residual_norm(ops.ADD_NORMED, kept, y, post, 1e-6, want, post)
    normed = ops.normed_rows(x, y, post, 1e-6, torch.empty_like(want), post, reader)
    assert type(normed) is ops.NormedRows and normed.product(w, rows // 2 if gated else rows, 2 if gated else 0) is None
    out, stream = reader(normed), ops.stream_behind(normed, x)
    assert stream is x and torch.equal(x, kept) and torch.equal(out, product(want, w))


@pytest.mark.parametrize("where", ["x", "y", "parts", "post", "next", "weight"])
@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan")])
@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_values_that_are_no_numbers(where, value, second, act):
    """Where the norm and the product one by one leave infinities and NaN; the other row and the other columns are not touched."""
    if where == "next" and not second:
        pytest.skip("no second norm")
    torch.manual_seed(2)
    T, K, N = 2, 1024, 96
    x, y, post, nxt = torch.randn(T, K, device="cuda"), torch.randn(2, T, K, device="cuda"), torch.rand(K, device="cuda") + 0.5, torch.rand(K, device="cuda") + 0.5
    w = (torch.randn(2 * N if act == 2 else N, K, device="cuda") * K ** -0.5).to(BF16)
    if where == "parts":
        y[0, 1, 77], y[1, 1, 77] = value, -value
    else:
        {"x": x[1], "y": y[1, 1], "post": post, "next": nxt, "weight": w[5]}[where][77] = value
    nxt = nxt if second else None
    kept, h = x.clone(), torch.empty(T, K, dtype=BF16, device="cuda")
    ops.residual_norm(ops.ADD_NORMED, kept, y, post, 1e-6, h, nxt)
    want = ops.linear_silu_gate(h, w) if act == 2 else ops.linear(h, w, "relu_squared" if act else None)
    rows = ops.NormedRows(x, y, post, nxt, 1e-6, torch.empty_like(h), torch.empty_like(x))
    got = rows.product(w, N, act)
    assert got is not None
    for one, other in ((rows.stream, kept), (got.float(), want.float())):
        assert torch.equal(one.isnan(), other.isnan()) and torch.equal(one.isinf(), other.isinf())
        finite = other.isfinite()          # (of these a row's last bits may turn: another order of its sums)
        assert torch.equal(one[other.isinf()], other[other.isinf()])
        assert not bool(finite.any()) or bool(((one - other).abs() <= 2.0 ** -6 * other[finite].abs().max())[finite].all())
    if where in ("x", "y", "parts"):
        assert bool(got[0].isfinite().all()) and bool(rows.stream[0].isfinite().all())
    if where == "weight":
        assert bool(got[:, [c for c in range(N) if c != 5]].isfinite().all())
