"""A residual norm and the product behind it in one launch, against float64: edges of its sizes, both forms of y, with and without the second norm."""
import pytest
import torch

from electrock_infer_amd import _lib
from electrock_infer_amd.layers import decoder_ops as ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("K,N,act", [(512, 1, 0), (512, 40, 1), (512, 24, 2), (1024, 4096, 0), (1536, 4097, 0), (2048, 8208, 1), (2048, 4104, 2),
                                     (2560, 16384, 0), (4096, 12288, 1), (4096, 8192, 2), (3584, 100, 2)])
@pytest.mark.parametrize("parts,second", [(0, True), (1, False), (4, True), (7, False)])
def test_one_launch_is_the_norm_and_the_product(T, K, N, act, parts, second):
    g = torch.Generator().manual_seed(K + N + parts)
    rand = lambda *shape: torch.randn(*shape, generator=g)
    x, post, nxt = rand(T, K), rand(K), rand(K) if second else None
    y = rand(T, K).to(BF16) if parts == 0 else rand(parts, T, K)
    w = (rand(2 * N if act == 2 else N, K) * K ** -0.5).to(BF16)
    dev = lambda t: None if t is None else t.cuda()
    dx, dy, dp, dn, dw = map(dev, (x, y, post, nxt, w))
    rows = ops.NormedRows(dx, dy, dp, dn, 1e-6, torch.empty(T, K, dtype=BF16, device="cuda"), torch.empty_like(dx))
    lib, out = _lib.load_decoder(), torch.full((T, N), float("nan"), dtype=BF16, device="cuda")
    assert lib.ed_norm_gemm_supported(T, N, K, act) == 1
    code = lib.ed_norm_gemm(dx.data_ptr(), dy.data_ptr(), _lib.dtype_code(dy.dtype), max(parts, 1), dp.data_ptr(), ops._ptr(dn), rows.spare.data_ptr(),
                            dw.data_ptr(), out.data_ptr(), T, N, K, act, 1e-6, _lib.current_stream(dx.device))
    assert code == 0
    norm = lambda v: v / (v.square().mean(-1, keepdim=True) + 1e-6).sqrt()
    y64 = y.double() if parts == 0 else y.double().sum(0)
    x64 = x.double() + norm(y64) * post.double()
    h = norm(x64) * nxt.double() if second else x64
    # float32: the parts' sum (2^-24 of all that it adds up, once a part), sixteen roundings of the mean, the root and the factors, the last sum
    parts_sum = (y.double() if parts == 0 else y.double().abs().sum(0)).abs()
    scale = post.double().abs() / (y64.square().mean(-1, keepdim=True) + 1e-6).sqrt()
    bound = 2.0 ** -24 * (x64.abs() + (16 * y64.abs() + max(parts, 1) * parts_sum) * scale)
    assert ((rows.spare.cpu().double() - x64).abs() <= bound).all()
    assert torch.equal(dx.cpu(), x)
    z, wd = h @ w.double().t(), w.double()
    # h is rounded to bf16 (eight significant bits): K independent errors of at most 2^-8 |h|, six standard deviations of their sum; the float32
    # sum beside them is nothing.  The result is rounded once more.
    e = 6 * 2.0 ** -8 / 3 ** 0.5 * (h.square() @ wd.square().t()).sqrt()
    if act == 2:
        gate, up, eg, eu = z[:, :N], z[:, N:], e[:, :N], e[:, N:]
        want, e = gate * torch.sigmoid(gate) * up, 1.1 * eg * (up.abs() + eu) + (gate * torch.sigmoid(gate)).abs() * eu
    elif act == 1:
        want, e = z.clamp(min=0).square(), 2 * z.abs() * e + e * e
    else:
        want = z
    assert ((out.cpu().double() - want).abs() <= e + 2.0 ** -8 * (want.abs() + e)).all()


@pytest.mark.parametrize("T,K", [(1, 2048), (2, 1024), (3, 2048), (1, 1000)])
def test_rows_reach_the_product_either_way(T, K):
    """A reader's hook, more rows and other widths get the rows themselves; the stream is the same wherever it lies."""
    torch.manual_seed(T + K)
    x, y, post = torch.randn(T, K, device="cuda"), torch.randn(2, T, K, device="cuda"), torch.rand(K, device="cuda") + 0.5
    w = (torch.randn(512, K, device="cuda") * K ** -0.5).to(BF16)
    kept, want = x.clone(), torch.empty(T, K, dtype=BF16, device="cuda")
    ops.residual_norm(ops.ADD_NORMED, kept, y, post, 1e-6, want, post)

    class Reader(torch.nn.Module):
        takes_normed_rows = True

        def forward(self, rows):
            return ops.linear(rows, w)

    for watched in (False, True):
        reader, seen = Reader(), []
        if watched:
            reader.register_forward_pre_hook(lambda module, args: seen.append(args[0]))
        mine = x.clone()
        rows = ops.normed_rows(mine, y, post, 1e-6, torch.empty_like(want), post, reader)
        assert (type(rows) is ops.NormedRows) == (not watched and T <= 2 and K % 512 == 0)
        out, stream = reader(rows), ops.stream_behind(rows, mine)
        if watched:
            assert torch.equal(seen[0], want)
        assert (stream - kept).abs().max() <= 2.0 ** -22 * kept.abs().max()
        assert (out.float() - ops.linear(want, w).float()).abs().max() <= 2.0 ** -6 * out.float().abs().max()      # (a row's last bit may turn)


@pytest.mark.parametrize("change", ["subclass", "object", "projection", "none"])
def test_a_forward_of_ones_own_gets_a_tensor(change):
    from electrock_infer_amd.layers.attention import SoftmaxAttention
    from electrock_infer_amd.layers.dense_mlp import DenseMLP
    x, y, w = torch.randn(1, 1024, device="cuda"), torch.randn(2, 1, 1024, device="cuda"), torch.ones(1024, device="cuda")

    class Own(DenseMLP):
        def forward(self, h):
            return super().forward(h * 1)

    if change == "projection":
        reader = SoftmaxAttention(1024, 8, 2, 64, 64, 1.0, 1e-6, BF16)
        reader.in_proj = torch.nn.Linear(1024, 768)
    else:
        reader = (Own if change == "subclass" else DenseMLP)(1024, 512, BF16)
        if change == "object":
            reader.forward = lambda h: h * 1
    rows = ops.normed_rows(x, y, w, 1e-6, torch.empty(1, 1024, dtype=BF16, device="cuda"), None, reader)
    assert (type(rows) is ops.NormedRows) == (change == "none")
