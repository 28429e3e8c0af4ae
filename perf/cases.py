"""Performance cases: what users of this package have it do, through its public entry points.

Two kinds of calls.  "layer": one Mixtral MoE layer, as an engine calls it once per decoder layer -- ``fused_experts`` with
router logits, or ``PostAttentionMoE`` (norm, gate, router and experts), on the 8x7B and 8x22B shapes, with the float32
result that the layer's tolerance is defined on or the bfloat16 one of the drop-in module.  "model": one step of the engine's
runner (batch preparation, forward pass, greedy token on the host) on a Nunivik or Feguvik model of eight layer runs, the
sizes of this repository's decoder benchmark: decode steps behind cached contexts, whole prompts, ragged batches of prompts,
and a portion of a prompt behind its earlier ones.  bfloat16 throughout, the type both are served in (float32 models exist to
check bfloat16 ones).
"""
import math

import torch

from electrock_infer_amd import PostAttentionMoE, MixtralMoE, RMSNorm, fused_experts
from electrock_infer_amd.harness import FeguvikConfig, LLMEngine, NunivikConfig, SamplingParams
from electrock_infer_amd.harness.feguvik import LayerSpec, LoopSpec
from electrock_infer_amd.harness.nunivik import MixerSpec
from electrock_infer_amd.harness.sequence import Sequence

DEVICE = "cuda"
SHAPES = {"8x7b": (4096, 14336), "8x22b": (6144, 16384)}      # hidden size, intermediate size of an expert
EXPERTS, TOP_K = 8, 2
NORM_EPS = {"layer": 1e-5, "model": 1e-6}
BLOCK, VOCAB = 32, 32000                                      # tokens of a cache block


def layer(name, shape, tokens, routing, form):
    return {"name": name, "kind": "layer", "shape": shape, "tokens": tokens, "routing": routing, "form": form}


def model(name, arch, width, seqs, tokens, past, ragged):
    """``seqs`` portions of (at most) ``tokens`` tokens behind (about) ``past`` computed ones."""
    return {"name": name, "kind": "model", "arch": arch, "width": width, "seqs": seqs, "tokens": tokens, "past": past, "ragged": ragged}


def listed():
    return [
        # one user's decode step: two experts' weights, four launches
        layer("moe_8x7b_t1", "8x7b", 1, "normal", "experts"),
        # the headline decode batch: every expert is streamed once
        layer("moe_8x7b_t64", "8x7b", 64, "normal", "experts"),
        # a busy server's mixed step, an odd batch with popular experts, the decoder layer's whole tail
        layer("moe_8x7b_t333_zipf", "8x7b", 333, "zipf", "tail"),
        # a full prefill batch
        layer("moe_8x7b_t8192", "8x7b", 8192, "normal", "experts"),
        # the large model, a prompt of odd length
        layer("moe_8x22b_t1501", "8x22b", 1501, "normal", "tail"),
        # generating for one user: latency and launches
        model("nunivik_2048_decode_1", "nunivik", 2048, 1, 1, 1023, False),
        # generating for many: weights, states and pages are streamed
        model("nunivik_2048_decode_64", "nunivik", 2048, 64, 1, 1024, True),
        # one long prompt
        model("nunivik_2048_prompt_8192", "nunivik", 2048, 1, 8192, 0, False),
        # several prompts of different lengths in one step, the wide model
        model("nunivik_4096_prompts_5x701", "nunivik", 4096, 5, 701, 0, True),
        # a batch that is no size of the recorded graphs, the wide model, longer contexts
        model("feguvik_4096_decode_23", "feguvik", 4096, 23, 1, 2000, True),
        # the prefill batch of eight equal prompts
        model("feguvik_2048_prompts_8x1024", "feguvik", 2048, 8, 1024, 0, False),
        # a later portion of one prompt, short
        model("feguvik_2048_portion_300", "feguvik", 2048, 1, 300, 1000, False),
    ]


def draw(rng):
    spread = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    most = max(cost(c) for c in listed())
    while True:
        if rng.random() < 0.4:
            case = layer("", rng.choice(["8x7b", "8x7b", "8x22b"]), spread(1, 8192), rng.choice(["normal", "zipf"]),
                         rng.choice(["experts", "tail"]))
        else:
            arch, width, ragged = rng.choice(["nunivik", "feguvik"]), rng.choice([2048, 4096]), rng.random() < 0.5
            if rng.random() < 0.5:
                case = model("", arch, width, spread(1, 64), 1, spread(32, 4000), ragged)
            else:
                seqs = spread(1, 8)
                case = model("", arch, width, seqs, spread(20, 8192 // seqs), rng.choice([0, 0, spread(32, 2000)]), ragged)
        del case["name"]
        if cost(case) <= most:
            return case


def cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


# ---- sizes of a case ----
def portions(case):
    """(tokens fed, tokens computed before) of every sequence; ragged ones between half and all of the case's numbers."""
    out = []
    for i in range(case["seqs"]):
        cut = lambda n, step: n - (i * step) % (n // 2 + 1) if case["ragged"] else n
        out.append((cut(case["tokens"], 131), cut(case["past"], 89)))
    return out


def specs(arch, width):
    """(kind, sizes of the mixer, feed-forward rows) of the eight layer runs' layers."""
    heads = width // 128
    if arch == "feguvik":
        gla = ("gla", {"heads": heads, "dim": 64, "vdim": 128, "tau": 16.0, "rank": 16}, 3 * width)
        latent = ("latent_attention", {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512,
                                       "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5}, 3 * width)
        return [gla, latent] * 3
    attention = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 30.0, "v_mix": True,
                 "rot": {"base": 10000.0, "dims": 128, "scaling": {"factor": 2.0}}}
    return [("delta", {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4}, 2 * width),
            ("attention", attention, 2 * width),
            ("mamba2", {"heads": 2 * width // 64, "groups": 1, "state": 128, "vdim": 64, "conv": 4, "norm_groups": 1}, 2 * width),
            ("attention", {**attention, "mask": {"size": 1024}}, 2 * width)] * 2


LOOP = (1, 3, 2)              # feguvik: layers 1 and 2 run twice
SIDE = 64                     # feguvik: per-layer token input


def runs(arch, width):
    """Layers in running order."""
    if arch == "nunivik":
        return list(range(8))
    start, stop, times = LOOP
    return list(range(start)) + list(range(start, stop)) * times + list(range(stop, 6))


def tensor_shapes(arch, width):
    """Checkpoint tensor -> shape."""
    W, t = width, {"embed": (VOCAB, width), "head": (VOCAB, width), "final.norm": (width,)}
    if arch == "feguvik":
        t.update({"side.embed": (VOCAB, 6 * SIDE), "loop.in": (W, 2 * W), "loop.step": (LOOP[2], W)})
    for i, (kind, m, ff) in enumerate(specs(arch, width)):
        p, x, H, v = f"l{i}.", f"l{i}.mix.", m["heads"], m["vdim"]
        t[p + "norm1"] = t[p + "norm2"] = (W,)
        if kind == "attention":
            G, d = m["kv_heads"], m["dim"]
            t.update({x + "q": (H * d, W), x + "k": (G * d, W), x + "v": (G * v, W), x + "q.norm": (d,), x + "k.norm": (d,), x + "vmix": ()})
        elif kind == "delta":
            G, d, taps = m["kv_heads"], m["dim"], m["conv"]
            t.update({x + "q": (G * d, W), x + "k": (G * d, W), x + "v": (H * v, W), x + "g": (H * v, W), x + "a": (H, W), x + "b": (H, W),
                      x + "q.conv": (G * d, taps), x + "k.conv": (G * d, taps), x + "v.conv": (H * v, taps), x + "norm": (v,),
                      x + "A_log": (H,), x + "dt_bias": (H,)})
        elif kind == "mamba2":
            n, taps = m["groups"] * m["state"], m["conv"]
            t.update({x + "in": (2 * H * v + 2 * n + H, W), x + "conv": (H * v + 2 * n, taps), x + "conv.b": (H * v + 2 * n,), x + "D": (H,),
                      x + "norm": (H * v,), x + "A_log": (H,), x + "dt_bias": (H,)})
        elif kind == "gla":
            d, r = m["dim"], m["rank"]
            t.update({x + "q": (H * d, W), x + "k": (H * d, W), x + "v": (H * v, W), x + "g": (H * v, W), x + "a1": (r, W),
                      x + "a2": (H * d, r), x + "a2.b": (H * d,), x + "norm": (v,)})
        else:
            d, r, c = m["dim"], m["rot_dim"], m["kv_rank"]
            t.update({x + "q": (H * (d + r), W), x + "dkv": (c + r, W), x + "dkv.norm": (c,), x + "uk": (H * d, c), x + "uv": (H * v, c),
                      x + "sink": (H,)})
        t[x + "o"] = (W, H * v)
        if arch == "feguvik":
            t.update({p + "norm1b": (W,), p + "ls1": (W,), p + "norm2b": (W,), p + "ls2": (W,), p + "mlp.up": (ff, W), p + "mlp.down": (W, ff),
                      p + "side.gate": (SIDE, W), p + "side.proj": (W, SIDE), p + "side.norm": (W,)})
        else:
            t.update({p + "mlp.gate": (ff, W), p + "mlp.up": (ff, W), p + "mlp.down": (W, ff)})
    return t


def state_shapes(kind, m, blocks, slots):
    """Cache or state of one layer run, as the model holds it: pages, or state and the last projections per sequence."""
    H, v = m["heads"], m["vdim"]
    if kind == "attention":
        return [(blocks, BLOCK, m["kv_heads"] * (m["dim"] + v))]
    if kind == "latent_attention":
        return [(blocks, BLOCK, m["kv_rank"] + m["rot_dim"])]
    if kind == "gla":
        return [(slots, H, m["dim"], v)]
    d, G = (m["dim"], m["kv_heads"]) if kind == "delta" else (m["state"], m["groups"])
    return [(slots, H, d, v), (slots, m["conv"], 2 * G * d + H * v)]


def work(case):
    if case["kind"] == "layer":
        H, I = SHAPES[case["shape"]]
        T = case["tokens"]
        # experts that T independent tokens with two distinct choices each touch (exact for one token)
        active = EXPERTS * (1.0 - (1.0 - TOP_K / EXPERTS) ** T) if case["routing"] == "normal" else min(EXPERTS, TOP_K * T)
        rows = T * H * (2 + 4) + T * EXPERTS * 2 if case["form"] == "experts" else T * H * 2 * 4 + (EXPERTS + 1) * H * 2
        return {"bytes": active * 3 * H * I * 2 + rows, "flops": T * TOP_K * 6.0 * H * I}
    arch, W = case["arch"], case["width"]
    parts = portions(case)
    T, S = sum(n for n, _ in parts), len(parts)
    shapes, kinds = tensor_shapes(arch, W), specs(arch, W)
    size = lambda name: math.prod(shapes[name])
    inside = lambda i: sum(size(n) for n in shapes if n.startswith(f"l{i}.") and len(shapes[n]) == 2)
    fixed = size("loop.in") if arch == "feguvik" else 0
    weights = sum(inside(i) for i in range(len(kinds))) + size("head") + fixed
    moved = weights * 2 + T * (W + (6 * SIDE if arch == "feguvik" else 0)) * 2 + S * VOCAB * 4
    flops = 2.0 * (T * (sum(inside(i) for i in runs(arch, W)) + fixed * LOOP[2]) + S * size("head"))
    for i in runs(arch, W):
        kind, m, _ = kinds[i]
        if kind in ("attention", "latent_attention"):
            window = (m.get("mask") or {}).get("size") or 1 << 30
            seen = sum(min(a + t + 1, window) for n, a in parts for t in range(n))
            held = sum(n + min(a, window - 1) for n, a in parts)                      # context rows read
            row = math.prod(state_shapes(kind, m, 1, 1)[0][2:])
            moved += (held + T) * row * 2
            flops += 2.0 * seen * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m["vdim"])
        else:
            shape = state_shapes(kind, m, 1, S)[0]
            moved += sum((1 if a == 0 else 2) for _, a in parts) * math.prod(shape[1:]) * 4
            flops += T * math.prod(shape[1:]) * (6.0 if kind == "delta" else 4.0)
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    """About four times the distance from ``exact`` that was measured: the layer's float32 result 2.9e-4 (fp16 activations), its
    bfloat16 one 1.8e-3; of a model the logits and the last layers' pages 1.5e-2 to 3e-2 (bfloat16 activations through eight
    layer runs), states less."""
    if case["kind"] == "layer":
        return {"rel": 1.2e-3 if case["form"] == "experts" else 8e-3}
    return {"rel": 9e-2}


# ---- inputs ----
def generator(seed, stream=0):
    return torch.Generator(device=DEVICE).manual_seed(seed * 1000 + stream)


def normal(g, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device=DEVICE).mul_(std).add_(mean).to(dtype)


def layer_inputs(case, seed):
    """Weights N(0, 0.02), rows N(0, 1), router logits N(0, 1); 'zipf' adds a bias that falls with the expert's rank."""
    H, I = SHAPES[case["shape"]]
    T, g = case["tokens"], generator(seed)
    w13 = torch.empty(EXPERTS, 2 * I, H, dtype=torch.bfloat16, device=DEVICE)
    w2 = torch.empty(EXPERTS, H, I, dtype=torch.float16, device=DEVICE)        # as the layer's loader keeps it
    for e in range(EXPERTS):
        w13[e] = normal(g, 2 * I, H, std=0.02)
        w2[e] = normal(g, H, I, std=0.02).to(torch.float16)
    zipf = -1.2 * torch.log(torch.arange(1, EXPERTS + 1, device=DEVICE, dtype=torch.float32)) if case["routing"] == "zipf" else 0.0
    s = {"w13": w13, "w2": w2, "x": normal(g, T, H)}
    if case["form"] == "experts":
        s["logits"] = (torch.randn(T, EXPERTS, generator=g, device=DEVICE) + zipf).to(torch.bfloat16)
    else:
        # a bias through the gate: one direction of the rows that every token has a share of
        gate = torch.randn(EXPERTS, H, generator=g, device=DEVICE) / math.sqrt(H)
        if case["routing"] == "zipf":
            s["x"][:, 0] = 8.0
            gate[:, 0] = zipf / 5.6
        s.update(gate=gate.to(torch.bfloat16), residual=normal(g, T, H), norm=normal(g, H, std=0.1, mean=1.0))
        if case["routing"] == "zipf":
            s["residual"][:, 0], s["norm"][0] = 0.0, 1.0
    return s


def model_weights(case, seed):
    """bfloat16 tensors under the checkpoint's names: matrices that keep a row's size, norms around one, decays that reach
    from a few tokens to hundreds, scores that are not flat, values mixed by a half."""
    g, out = generator(seed), {}
    around = {"vmix": (0.5, 0.1), "q.norm": (1.7, 0.2), "k.norm": (1.5, 0.2), "A_log": (-1.0, 1.0), "dt_bias": (-2.0, 1.5),
              "sink": (0.5, 1.0), "a2.b": (2.0 + math.log(17.0), 1.5), "conv.b": (0.0, 0.1)}
    for name, shape in tensor_shapes(case["arch"], case["width"]).items():
        if name in ("embed", "side.embed"):
            mean, std = 0.0, 1.0
        elif name == "loop.step":
            mean, std = 0.0, 0.3
        elif name.endswith("conv"):
            mean, std = 0.3, 0.5
        elif len(shape) == 2:
            mean, std = 0.0, (2.0 if case["arch"] == "feguvik" and name.endswith("mix.q") else 1.0) / math.sqrt(shape[1])
        else:
            mean, std = next((v for k, v in around.items() if name.endswith(k)), (1.0, 0.1))
        out[name] = normal(g, *shape, std=std, mean=mean)
    return out


def model_inputs(case, seed):
    """Tokens, pages and earlier state of every sequence.  The pages of a long-lived cache lie in any order."""
    g, parts = generator(seed, 1), portions(case)
    pages = [-(-(n + a) // BLOCK) for n, a in parts]
    order = torch.randperm(sum(pages), generator=g, device=DEVICE).tolist()
    tables = [order[sum(pages[:i]):sum(pages[:i + 1])] for i in range(len(pages))]
    tokens = [torch.randint(0, VOCAB, (n + a,), generator=g, device=DEVICE).tolist() for n, a in parts]
    kinds, caches = specs(case["arch"], case["width"]), []
    for i in runs(case["arch"], case["width"]):
        kind, m, _ = kinds[i]
        shapes = state_shapes(kind, m, len(order), len(parts))
        if kind in ("attention", "latent_attention"):
            caches.append([normal(g, *shapes[0])])                               # keys and latents are normed rows
        else:
            caches.append([normal(g, *shapes[0], std=0.5, dtype=torch.float32)] + [normal(g, *s) for s in shapes[1:]])
    return parts, tables, tokens, caches


def prepare(case, seed):
    if case["kind"] == "layer":
        s = layer_inputs(case, seed)
        if case["form"] == "tail":
            H, I = SHAPES[case["shape"]]
            with torch.device("meta"):
                moe = MixtralMoE(EXPERTS, TOP_K, H, I, params_dtype=torch.bfloat16)
                norm = RMSNorm(H, NORM_EPS["layer"])
            hold = lambda t: torch.nn.Parameter(t, requires_grad=False)
            moe.gate.weight, moe.experts.w13_weight, moe.experts.w2_weight = hold(s["gate"]), hold(s["w13"]), hold(s["w2"])
            norm.weight = hold(s["norm"])
            s["tail"] = PostAttentionMoE(norm, moe)
        return s
    parts, tables, tokens, caches = model_inputs(case, seed)
    kinds, width = specs(case["arch"], case["width"]), case["width"]
    if case["arch"] == "nunivik":
        cfg = NunivikConfig(vocab_size=VOCAB, width=width, layers=[MixerSpec(k, m, ff) for k, m, ff in kinds], norm_eps=NORM_EPS["model"])
    else:
        cfg = FeguvikConfig(vocab_size=VOCAB, width=width, layers=[LayerSpec(k, m, ff, m.get("rank", 0)) for k, m, ff in kinds],
                            norm_eps=NORM_EPS["model"], side_dim=SIDE, loop=LoopSpec(*LOOP))
    engine = LLMEngine(cfg, max_model_len=16384, max_num_seqs=len(parts), max_num_batched_tokens=16384, kvcache_block_size=BLOCK,
                       num_kvcache_blocks=sum(len(t) for t in tables), reuse_prefix=False)
    net = engine.model_runner.model
    for name, tensor in model_weights(case, seed).items():
        target, section = net.checkpoint_target(name)
        param = net.get_parameter(target)
        if section is None:
            param.data.copy_(tensor)
        else:
            param.weight_loader(param, tensor, section)
    net.finish_loading()
    seqs = []
    for i, (n, a) in enumerate(parts):
        s = Sequence(tokens[i], SamplingParams(temperature=0.0, max_tokens=1 << 20, ignore_eos=True))
        s.block_table, s.state_slot, s.num_computed_tokens, s.num_scheduled_tokens = tables[i], i, a, n
        seqs.append(s)
    held = []                              # the sequences' part of every cache
    for cache, values in zip(net.caches, caches):
        for t, v in zip(cache if isinstance(cache, tuple) else (cache,), values):
            t[:len(v)].copy_(v)
            held.append(t[:len(v)])
    return {"engine": engine, "seqs": seqs, "prefill": case["tokens"] > 1, "caches": held}


def run(state):
    if "engine" in state:
        _, logits = state["engine"].model_runner.run(state["seqs"], state["prefill"], return_logits=True)
        return {"logits": logits, "caches": state["caches"]}
    if "tail" in state:
        return state["tail"](state["x"], state["residual"])
    return fused_experts(state["x"], state["w13"], state["w2"], state["logits"], TOP_K, out_dtype=torch.float32)


# ---- the same in 64 bits ----
def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(x):
    return x * torch.sigmoid(x)


def layer_exact(case, seed):
    s = layer_inputs(case, seed)
    x, residual = s["x"].double(), None
    if case["form"] == "tail":
        # the module's rounding points: the sum and the normed rows are the layer's inputs and outputs in bfloat16
        residual = x + s["residual"].double()
        x = (rms(residual, NORM_EPS["layer"])).to(torch.bfloat16).double() * s["norm"].double()
        x = x.to(torch.bfloat16).double()
        logits = (x @ s["gate"].double().t()).float().to(torch.bfloat16).double()
    else:
        logits = s["logits"].double()
    p = torch.softmax(logits, -1)
    # the largest ones, the lower index first where two are equal
    ids = torch.sort(logits, dim=-1, descending=True, stable=True).indices[:, :TOP_K]
    weight = p.gather(1, ids)
    weight = weight / weight.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    I = s["w2"].shape[2]
    for e in range(EXPERTS):
        row, place = (ids == e).nonzero(as_tuple=True)
        if row.numel() == 0:
            continue
        w13 = s["w13"][e].double()
        u = silu(x[row] @ w13[:I].t()) * (x[row] @ w13[I:].t())
        del w13
        out.index_add_(0, row, (u @ s["w2"][e].double().t()) * weight[row, place][:, None])
    return out if residual is None else (out, residual)


def turn(x, positions, dims, base, factor, halves):
    """Rotation of pairs of the first ``dims`` elements: neighbours, or element i with i + dims / 2."""
    i = torch.arange(dims // 2, device=x.device, dtype=torch.float64)
    # (frequencies are constants of the model, held in float32)
    angle = positions[:, None] * (base ** (-2.0 * i / dims) / factor).float().double()
    angle = angle.view(len(positions), *[1] * (x.dim() - 2), -1)
    c, s = torch.cos(angle), torch.sin(angle)
    out = x.clone()
    u, v = (x[..., :dims // 2], x[..., dims // 2:dims]) if halves else (x[..., 0:dims:2], x[..., 1:dims:2])
    a, b = u * c - v * s, v * c + u * s
    if halves:
        out[..., :dims] = torch.cat([a, b], -1)
    else:
        out[..., :dims] = torch.stack([a, b], -1).flatten(-2)
    return out


class ExactModel:
    """One step of a model on plain float64 tensors: linear parts on all tokens, mixers sequence by sequence."""

    def __init__(self, case, seed):
        self.case, self.arch, self.width, self.eps = case, case["arch"], case["width"], NORM_EPS["model"]
        self.w = model_weights(case, seed)
        self.parts, self.tables, tokens, self.caches = model_inputs(case, seed)
        self.new, at = [], 0              # rows of a sequence's new tokens
        for n, a in self.parts:
            self.new.append(slice(at, at + n))
            at += n
        self.tokens = torch.tensor([t for s, (n, a) in zip(tokens, self.parts) for t in s[a:]], device=DEVICE)
        self.positions = [torch.arange(a, a + n, device=DEVICE, dtype=torch.float64) for n, a in self.parts]
        self.rows = [(torch.tensor(t, device=DEVICE)[:, None] * BLOCK + torch.arange(BLOCK, device=DEVICE)).flatten()[:n + a]
                     for t, (n, a) in zip(self.tables, self.parts)]
        self.caches = [[t.double() for t in c] for c in self.caches]
        self.carried = None

    def mat(self, x, name):
        return x @ self.w[name].double().t()

    def vec(self, name):
        return self.w[name].double()

    def attend(self, q, k, v, scale, cap, window, sink, past):
        """q [n, heads, d], k [m, groups, d], v [m, groups, e] -> [n, heads, e]; the first query is position ``past``."""
        n, m, share = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
        out = torch.empty(n, q.shape[1], v.shape[2], dtype=torch.float64, device=q.device)
        for at in range(0, n, 2048):
            to = min(n, at + 2048)
            gap = torch.arange(past + at, past + to, device=q.device)[:, None] - torch.arange(m, device=q.device)
            hide = (gap < 0) | (gap >= window)
            for h in range(q.shape[1]):
                s = q[at:to, h] @ k[:, h // share].t() * scale
                s = (cap * torch.tanh(s / cap) if cap else s).masked_fill_(hide, -math.inf)
                if sink is not None:
                    s = torch.cat([s, sink[h].expand(to - at, 1)], 1)
                out[at:to, h] = torch.softmax(s, -1)[:, :m] @ v[:, h // share]
        return out

    def attention(self, h, r, x, m):
        H, G, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        T, pages = h.shape[0], self.caches[r][0].view(-1, G * (d + e))
        pos = torch.cat(self.positions)
        rot = lambda t: turn(t, pos, m["rot"]["dims"], m["rot"]["base"], m["rot"]["scaling"]["factor"], False)
        q = rot(rms(self.mat(h, x + "q").view(T, H, d), self.eps) * self.vec(x + "q.norm"))
        k = rot(rms(self.mat(h, x + "k").view(T, G, d), self.eps) * self.vec(x + "k.norm"))
        v = self.mat(h, x + "v")
        if self.carried is None:
            self.carried = v
        else:
            v = (1.0 - self.vec(x + "vmix")) * v + self.vec(x + "vmix") * self.carried
        out = torch.empty(T, H, e, dtype=torch.float64, device=h.device)
        window = (m.get("mask") or {}).get("size") or 1 << 30
        for new, rows, (n, a) in zip(self.new, self.rows, self.parts):
            pages[rows[a:]] = torch.cat([k[new].flatten(1), v[new]], 1)
            kv = pages[rows]
            out[new] = self.attend(q[new], kv[:, :G * d].view(-1, G, d), kv[:, G * d:].view(-1, G, e), m["scale"], m["softcap"], window, None, a)
        return self.mat(out.flatten(1), x + "o")

    def latent_attention(self, h, r, x, m):
        H, d, rot, e, c = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        T, pages, pos = h.shape[0], self.caches[r][0].view(-1, c + rot), torch.cat(self.positions)
        q = self.mat(h, x + "q").view(T, H, d + rot)
        q = torch.cat([q[..., :d], turn(q[..., d:], pos, rot, m["rot"]["base"], 1.0, True)], -1)
        down = self.mat(h, x + "dkv")
        row = torch.cat([rms(down[:, :c], self.eps) * self.vec(x + "dkv.norm"), turn(down[:, c:], pos, rot, m["rot"]["base"], 1.0, True)], -1)
        out = torch.empty(T, H, e, dtype=torch.float64, device=h.device)
        for new, rows, (n, a) in zip(self.new, self.rows, self.parts):
            pages[rows[a:]] = row[new]
            kv = pages[rows]
            k = torch.cat([self.mat(kv[:, :c], x + "uk").view(-1, H, d), kv[:, None, c:].expand(-1, H, -1)], -1)
            v = self.mat(kv[:, :c], x + "uv").view(-1, H, e)
            out[new] = self.attend(q[new], k, v, m["scale"], 0.0, 1 << 30, self.vec(x + "sink"), a)
        return self.mat(out.flatten(1), x + "o")

    def gla(self, h, r, x, m):
        H, d, e = m["heads"], m["dim"], m["vdim"]
        T = h.shape[0]
        q, k, v = (self.mat(h, x + s).view(T, H, -1) for s in "qkv")
        q = q * d ** -0.5
        z = self.mat(self.mat(h, x + "a1"), x + "a2") + self.vec(x + "a2.b")
        decay = torch.sigmoid(z).pow(1.0 / m["tau"]).view(T, H, d, 1)
        out = torch.empty(T, H, e, dtype=torch.float64, device=h.device)
        for i, (new, (n, a)) in enumerate(zip(self.new, self.parts)):
            S = self.caches[r][0][i] if a else torch.zeros(H, d, e, dtype=torch.float64, device=h.device)
            for t in range(new.start, new.stop):
                S = torch.addcmul(k[t, :, :, None] * v[t, :, None, :], decay[t], S)
                out[t] = torch.bmm(q[t, :, None, :], S)[:, 0]
            self.caches[r][0][i] = S
        g = self.mat(h, x + "g")
        return self.mat((rms(out, self.eps) * self.vec(x + "norm")).flatten(1) * silu(g), x + "o")

    def convolve(self, p, r, taps, bias):
        """SiLU of the causal convolution of every sequence's projections; the ring takes those that a later token needs."""
        K, ring, out = taps.shape[1], self.caches[r][1], torch.empty_like(p)
        for i, (new, (n, a)) in enumerate(zip(self.new, self.parts)):
            before = [ring[i, (a - K + 1 + j) % K] if a - K + 1 + j >= 0 else torch.zeros_like(ring[i, 0]) for j in range(K - 1)]
            every = torch.cat([torch.stack(before), p[new]])
            out[new] = sum(every[j:j + n] * taps[:, j] for j in range(K))
            for t in range(max(0, n - K + 1), n):
                ring[i, (a + t) % K] = p[new.start + t]
        return silu(out if bias is None else out + bias)

    def recur(self, r, q, k, v, decay, beta, delta):
        out = torch.empty_like(v)
        for i, (new, (n, a)) in enumerate(zip(self.new, self.parts)):
            S = self.caches[r][0][i] if a else torch.zeros_like(self.caches[r][0][i])
            for t in range(new.start, new.stop):
                S = S * decay[t]
                u = beta[t] * (v[t] - torch.bmm(k[t, :, None, :], S)[:, 0] if delta else v[t])
                S = torch.baddbmm(S, k[t, :, :, None], u[:, None, :])
                out[t] = torch.bmm(q[t, :, None, :], S)[:, 0]
            self.caches[r][0][i] = S
        return out

    def delta(self, h, r, x, m):
        H, G, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        T = h.shape[0]
        p = torch.cat([self.mat(h, x + s) for s in "qkv"], 1)
        q, k, v = torch.split(self.convolve(p, r, torch.cat([self.vec(x + s + ".conv") for s in "qkv"]), None), [G * d, G * d, H * e], 1)
        unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
        q, k = (unit(t.view(T, G, d)).repeat_interleave(H // G, 1).contiguous() for t in (q, k))
        beta = torch.sigmoid(self.mat(h, x + "b"))
        step = torch.nn.functional.softplus(self.mat(h, x + "a") + self.vec(x + "dt_bias"), threshold=1000.0)
        decay = torch.exp(-torch.exp(self.vec(x + "A_log")) * step)
        o = self.recur(r, q * d ** -0.5, k, v.view(T, H, e).contiguous(), decay[:, :, None, None], beta[:, :, None], True)
        o = rms(o, self.eps) * self.vec(x + "norm") * silu(self.mat(h, x + "g")).view(T, H, e)
        return self.mat(o.flatten(1), x + "o")

    def mamba2(self, h, r, x, m):
        H, e, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        T, inner = h.shape[0], H * e
        z, p, dt = torch.split(self.mat(h, x + "in"), [inner, inner + 2 * G * N, H], 1)
        # the checkpoint's order is x | B | C; the ring holds C | B | x
        order = lambda t: torch.cat([t[..., inner + G * N:], t[..., inner:inner + G * N], t[..., :inner]], -1)
        conv = self.vec(x + "conv")
        C, B, v = torch.split(self.convolve(order(p), r, order(conv.t()).t(), order(self.vec(x + "conv.b"))), [G * N, G * N, inner], 1)
        C, B = (t.view(T, G, N).repeat_interleave(H // G, 1).contiguous() for t in (C, B))
        dt = torch.nn.functional.softplus(dt + self.vec(x + "dt_bias"), threshold=1000.0)
        decay = torch.exp(-torch.exp(self.vec(x + "A_log")) * dt)
        v = v.reshape(T, H, e).contiguous()
        y = self.recur(r, C, B, v, decay[:, :, None, None], dt[:, :, None], False) + self.vec(x + "D")[:, None] * v
        y = (y.flatten(1) * silu(z)).view(T, m["norm_groups"], -1)
        return self.mat(rms(y, self.eps).flatten(1) * self.vec(x + "norm"), x + "o")

    def forward(self):
        x, kinds, norm = self.vec("embed")[self.tokens], specs(self.arch, self.width), lambda t, n: rms(t, self.eps) * self.vec(n)
        x0, passes = x, 0
        for r, i in enumerate(runs(self.arch, self.width)):
            kind, m, _ = kinds[i]
            p = f"l{i}."
            mix = getattr(self, kind)
            if self.arch == "nunivik":
                x = x + norm(mix(x, r, p + "mix.", m), p + "norm1")
                x = x + norm(self.mat(silu(self.mat(x, p + "mlp.gate")) * self.mat(x, p + "mlp.up"), p + "mlp.down"), p + "norm2")
                continue
            if i == LOOP[0]:
                x = self.mat(torch.cat([x, x0], 1), "loop.in") + self.vec("loop.step")[passes]
                passes += 1
            x = x + norm(mix(norm(x, p + "norm1"), r, p + "mix.", m), p + "norm1b") * self.vec(p + "ls1")
            u = torch.relu(self.mat(norm(x, p + "norm2"), p + "mlp.up"))
            x = x + norm(self.mat(u * u, p + "mlp.down"), p + "norm2b") * self.vec(p + "ls2")
            side = self.w["side.embed"][self.tokens][:, i * SIDE:(i + 1) * SIDE].double()
            g = torch.nn.functional.gelu(self.mat(x, p + "side.gate"), approximate="tanh") * side
            x = x + norm(self.mat(g, p + "side.proj"), p + "side.norm")
        last = torch.tensor([s.stop - 1 for s in self.new], device=DEVICE)
        return {"logits": self.mat(norm(x, "final.norm")[last], "head"), "caches": [t for c in self.caches for t in c]}


def exact(case, seed):
    with torch.no_grad():
        return layer_exact(case, seed) if case["kind"] == "layer" else ExactModel(case, seed).forward()
