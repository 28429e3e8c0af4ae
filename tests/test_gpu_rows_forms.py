"""The row norms in every form that the launch picks by rows and width, at its edges, with partial sums of every number."""
import pytest
import torch

from electrock_infer_amd.layers import decoder_ops as ops
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu
F32, BF16, EPS = torch.float32, torch.bfloat16, 1e-5
# one vector per thread up to 256 rows of 1028 .. 2048 / .. 4096, two and four beyond (with their loads at once or in turn), eight, 1024
# threads; rows that are no multiple of four go element by element
ROWS = [(1, 1024), (256, 1028), (257, 1028), (256, 2048), (256, 2052), (257, 2048), (257, 2052), (256, 4096), (257, 4096), (1024, 4096), (1025, 4096),
        (3, 4100), (2, 8192), (2, 8196), (3, 32768), (5, 1027), (3, 8191), (2, 8193)]


def rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def near(got, want, dtype):
    """float32 sums of a row in any order: some sqrt(W) 2^-24 of its size; a result in bf16: half a step, 2^-8 of a value."""
    got = got.double().cpu()
    bound = (1e-5 if dtype == F32 else 2.0 ** -8 + 1e-5) * want.abs() + 3e-6 * want.abs().max()
    assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() / bound).max())


@pytest.mark.parametrize("T,W", ROWS)
@pytest.mark.parametrize("y_dtype,dtype,parts", [(BF16, BF16, 1), (F32, F32, 1), (F32, BF16, 1), (F32, BF16, 2), (F32, BF16, 5), (F32, BF16, 6), (F32, F32, 9)])
def test_residual_norm(T, W, y_dtype, dtype, parts):
    announce(f"residual norm forms {T} {W} {y_dtype} {dtype} parts {parts}")
    g = torch.Generator(device="cuda").manual_seed(W + T + parts)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y, post, nxt = rand(T, W), rand(parts, T, W).to(y_dtype), rand(W), rand(W)
    whole = y.double().sum(0)
    for update in (ops.KEEP, ops.ADD_NORMED, ops.REPLACE):
        for p, n in ((post, nxt), (post, None)) + (((None, nxt),) if update == ops.REPLACE else ()):
            stream, out = x.clone(), torch.full((T, W + 4), 7.0, dtype=dtype, device="cuda")
            ops.residual_norm(update, stream, None if update == ops.KEEP else (y if parts > 1 else y[0]), p, EPS, out[:, :W], n)
            want = {ops.KEEP: x.double(), ops.ADD_NORMED: x.double() + rms(whole) * post.double(), ops.REPLACE: whole + (0.0 if p is None else p.double())}[update].cpu()
            near(stream, want, F32)
            near(out[:, :W], want if n is None else rms(want) * n.double().cpu(), dtype)
            assert bool((out[:, W:] == 7).all())
        stream = x.clone()
        if update != ops.KEEP:
            ops.residual_norm(update, stream, y if parts > 1 else y[0], post, EPS, None)
            near(stream, (x.double() + rms(whole) * post.double() if update == ops.ADD_NORMED else whole + post.double()).cpu(), F32)


# partial sums element by element: one piece of 16 elements a thread (256 threads up to 4096 columns), two, and the same of 1024 threads;
# more rows than are requested at once
@pytest.mark.parametrize("T,W", [(2, 4095), (2, 4097), (1, 8190), (2, 9001), (2, 16383), (2, 16385), (1, 32767), (300, 4096), (300, 2048)])
@pytest.mark.parametrize("dtype,parts", [(F32, 2), (BF16, 3), (F32, 8)])
def test_partial_sums_in_pieces(T, W, dtype, parts):
    test_residual_norm(T, W, F32, dtype, parts)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("T,parts,size", [(3, 1, 512), (3, 1, 516), (3, 1, 1024), (2, 3, 1028), (256, 1, 4096), (257, 1, 4096), (128, 2, 2048), (129, 2, 2048),
                                          (3, 1, 4100), (3, 1, 8192), (2, 1, 8196), (300, 1, 8192), (3, 2, 1021), (3, 1, 8191), (2, 1, 9001), (1, 1, 32768)])
def test_gated_norm(T, parts, size, dtype):
    announce(f"gated norm forms {T} {parts} {size} {dtype}")
    g = torch.Generator(device="cuda").manual_seed(size + T)
    y, z, w = (torch.randn(*s, generator=g, device="cuda") for s in ((T, parts * size), (T, parts * size + 4), (parts * size,)))
    y, z = y.to(dtype), z.to(dtype)
    v = y.double() * torch.nn.functional.silu(z[:, :parts * size].double())
    want = (rms(v.view(T, parts, size)).flatten(1) * w.double()).cpu()
    near(ops.gated_norm_(y, z.data_ptr(), z.stride(0), w, parts, EPS), want, dtype)


# many rows: loads at once up to 1024 elements, in turn beyond in bf16
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("T,parts,size", [(257, 1, 1024), (257, 1, 1028), (86, 3, 1028), (300, 1, 3000), (257, 1, 4100)])
def test_gated_norm_of_many_rows(T, parts, size, dtype):
    test_gated_norm(T, parts, size, dtype)
