"""Recurrences of prompts whose values no bf16 holds: infinities, and float32 numbers beyond the largest bf16.  The prompt kernels multiply
by float32 operands as sums of bf16 parts; what has no such parts comes out as float32 products give it.

The reference is the recurrence token by token in float64, on the kernels' own inputs (taps of one: the projections behind a SiLU)."""
import pytest
import torch

from electrock_infer_amd.harness import SamplingParams
from electrock_infer_amd.harness.batch import make_ragged
from electrock_infer_amd.harness.sequence import Sequence
from tests.gpu_util import DEV, announce
from tests.nunivik_util import delta, mamba
from tests.test_gpu_nunivik_ops import BLOCK, F32, N, recurrent, weights

pytestmark = pytest.mark.gpu
BEYOND = 3.399e38           # float32 reaches 3.4028e38, bf16 3.3895e38


class Case:
    """A mixer's recurrence on projections of its own, two sequences in one batch, the second untouched by what the first holds."""

    def __init__(self, entry, tokens, start=0):
        m = entry["mixer"]
        self.m, self.is_delta, self.start, self.tokens = m, entry["type"] == "delta", start, tokens
        self.H, self.G, self.dim, self.vdim = m["heads"], m.get("kv_heads", m.get("groups")), m.get("dim", m.get("state")), m["vdim"]
        w = weights(entry, 64, 1)
        w.update({k: torch.ones_like(t) for k, t in w.items() if k.endswith("conv")})
        w["mix.A_log"], w["mix.dt_bias"] = torch.full((self.H,), -4.0), torch.zeros(self.H)
        if "mix.conv.b" in w:
            w["mix.conv.b"].zero_()
        self.mix = recurrent(entry, 64, F32, w)
        self.p = torch.randn(2 * tokens, self.mix.in_proj.out_rows, generator=torch.Generator().manual_seed(2))
        self.states = torch.zeros(2, self.H, self.dim, self.vdim) if start == 0 else \
            torch.randn(2, self.H, self.dim, self.vdim, generator=torch.Generator().manual_seed(3))

    def section(self, name):
        at = self.mix.in_proj.offset[name]
        return self.p[:, at:at + self.mix.in_proj.rows[name]]

    def run(self, chunk):
        """(outputs, states) of the kernels, on the host."""
        Sequence.block_size, seqs = BLOCK, []
        for i in range(2):
            s = Sequence([0] * (self.start + self.tokens), SamplingParams())
            s.block_table, s.state_slot = list(range(s.num_blocks)), i
            s.num_computed_tokens, s.num_scheduled_tokens = self.start, self.tokens
            seqs.append(s)
        batch, cache = make_ragged(seqs, BLOCK, chunk, DEV), self.mix.new_cache(0, BLOCK, 2, DEV)
        cache.states.copy_(self.states)
        named = {"beta": "beta", "gate": "gate", "norm": self.mix.norm, "q_scale": self.dim ** -0.5, "unit_eps": 1e-6} if self.is_delta else {"skip": self.mix.skip}
        return self.mix.recur(self.p.to(DEV), batch, cache, **named).cpu(), cache.states.cpu()

    def want(self):
        """(outputs in front of norm and gate, states) in float64."""
        H, G, T = self.H, self.G, 2 * self.tokens
        part = lambda n: self.section(n).double()
        act = lambda n, *shape: N.silu(part(n)).view(T, *shape)
        share = torch.arange(H) // (H // G)
        q, k, v = act("q", G, self.dim)[:, share], act("k", G, self.dim)[:, share], act("v", H, self.vdim)
        step = N.softplus(part("decay"))
        decay, S = torch.exp(-torch.exp(torch.tensor(-4.0, dtype=torch.float64)) * step), self.states.double().clone()
        if self.is_delta:
            q, k, beta = N.unit(q) * self.dim ** -0.5, N.unit(k), torch.sigmoid(part("beta"))
        out = torch.empty(T, H, self.vdim, dtype=torch.float64)
        for i in range(2):
            for t in range(i * self.tokens, (i + 1) * self.tokens):
                s = S[i] * decay[t][:, None, None]
                u = beta[t][:, None] * (v[t] - (s * k[t][:, :, None]).sum(1)) if self.is_delta else (step[t][:, None] * v[t]).float().double()
                S[i] = s + k[t][:, :, None] * u[:, None, :]
                out[t] = (S[i] * q[t][:, :, None]).sum(1)
        return out, S


def close(got, want):
    """[..., rows, columns]: every column's finite values at a float32 recurrence's distance (hundreds of float32 sums: 1e-5), infinities
    where they are."""
    finite, got = torch.isfinite(want), got.double()
    assert torch.equal(torch.isfinite(got), finite) and torch.equal(got[~finite], want[~finite])
    a, b = (torch.where(finite, t, 0.0) / 2.0 ** 64 for t in (got, want))
    assert bool(((a - b).norm(dim=-2) <= 1e-5 * b.norm(dim=-2)).all())


# heads that share a workgroup, two pieces of a key per thread, a whole tile and ragged ones; one chunk and several
@pytest.mark.parametrize("entry", [mamba(4, 1, 128, 64, 1), mamba(2, 1, 24, 20, 1), mamba(1, 1, 200, 130, 1), mamba(2, 2, 64, 128, 1)],
                         ids=lambda e: "-".join(str(v) for v in e["mixer"].values()))
@pytest.mark.parametrize("chunk", [256, 64])
def test_infinite_update(entry, chunk):
    announce(f"recurrence range: infinite update {entry['mixer']} {chunk}")
    case = Case(entry, 150)
    case.section("v")[70, 3], case.section("decay")[70, 0] = 2.0 ** 127, 4.0       # (their product overflows)
    (out, states), (ref, want) = case.run(chunk), case.want()
    assert (~torch.isfinite(want)).sum() == case.dim
    close(states, want)
    ref += case.mix.skip.cpu().double()[:, None] * N.silu(case.section("v").double()).view(ref.shape)
    ref = ref.flatten(1)
    close(out[:64], ref[:64])                     # (in front of the block with the infinity)
    close(out[150:], ref[150:])
    others = torch.arange(ref.shape[1]) != 3      # (head 0, column 3)
    close(out[:, others], ref[:, others])


@pytest.mark.parametrize("entry", [mamba(4, 1, 128, 64, 1), mamba(2, 1, 24, 20, 1)], ids=lambda e: "-".join(str(v) for v in e["mixer"].values()))
@pytest.mark.parametrize("chunk", [256, 64])
def test_update_beyond_the_largest_bf16(entry, chunk):
    announce(f"recurrence range: update {entry['mixer']} {chunk}")
    case = Case(entry, 90)
    for n in "qk":
        case.section(n).mul_(1e-3)
    # the last token of a block, whose update no decay makes smaller: softplus(decay) times the value
    case.section("v")[47, 3] = 2.0 ** 127
    case.section("decay")[47, 0] = float(torch.log(torch.expm1(torch.tensor(BEYOND / 2.0 ** 127, dtype=torch.float64))))
    (_, states), (_, want) = case.run(chunk), case.want()
    assert torch.isfinite(want).all() and float(want.abs().max()) > 1e33
    close(states, want)


# an output pass of eight waves and one of sixteen, two pieces of a key per thread
@pytest.mark.parametrize("entry", [delta(4, 2, 128, 128, 1), delta(2, 1, 40, 24, 1), delta(1, 1, 64, 160, 1), delta(1, 1, 256, 64, 1)],
                         ids=lambda e: "-".join(str(v) for v in e["mixer"].values()))
@pytest.mark.parametrize("chunk", [256, 16])
def test_state_beyond_the_largest_bf16(entry, chunk):
    announce(f"recurrence range: state {entry['mixer']} {chunk}")
    case = Case(entry, 40, start=5)
    case.states[0, 0, 7, 5] = BEYOND
    (_, states), (_, want) = case.run(chunk), case.want()
    assert torch.isfinite(want).all() and float(want.abs().max()) > 1e37
    close(states, want)
    close(states[1], want[1])
