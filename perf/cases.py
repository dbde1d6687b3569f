"""What the speed of this framework is measured on: steps of whole models through ``ModelRunner``, as a program that serves or
scores requests takes them, in every architecture that is registered.

A case names a model (``family``, layer sizes ``size``, number of ``layers``, ``dtype``) and what its requests do:

  kind "next"      the requests hold ``tokens`` tokens of context between them; a pass is one decode step of all of them at these
                   contexts, with ``portion`` prompt tokens of one more request in the same step where that is not 0.  The step
                   writes the same cache entries in every pass.  Only models whose caches hold nothing but entries by position.
  kind "generate"  a pass is the requests' whole life: they are admitted, their prompts (``tokens`` between them, in portions of
                   up to ``portion`` tokens, at most 2,048 tokens a step) run, then each gets ``new`` given tokens one by one beside
                   whatever is still left of the others' prompts, and is finished.  ``new`` 0: prompts alone.

Outputs are the float32 logits of every wanted row: the last of each prompt and every decoded token.  Token ids are log-uniform,
which is close to how often words occur; lengths are ragged.  Routers get weights under which a token's experts follow from its
id with a margin, as a trained router's do: a choice between experts on the last bit of their logits would measure nothing.
"""
import math
import random
import re

import torch

from swifttransformer_amd.config.cache_param import CacheParam
from swifttransformer_amd.config.registry import hyper_param_by_name
from swifttransformer_amd.engine.step import ModelRunner, StepEntry
from swifttransformer_amd.models import build_model

PAGE = 16
BUDGET = 2048                   # tokens of a step
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
FAMILIES = ("opt", "zitupel", "zimorax", "gisedra", "pupalix", "fiterax", "fefozen")


def _case(name, family, size, layers, kind, requests, tokens, new=0, portion=BUDGET, dtype="bf16"):
    c = {"name": name, "family": family, "size": size, "layers": layers, "kind": kind, "requests": requests, "tokens": tokens,
         "new": new, "portion": portion, "dtype": dtype}
    return c if name else {k: v for k, v in c.items() if k != "name"}


def listed():
    return [
        # one user at a short context on the smallest model: all launches, almost no bytes
        _case("opt-125m next 1", "opt", "125m", 12, "next", 1, 97, portion=0),
        # the headline decode workload: 8 requests half way from 1,024-token prompts to the 2,048-token context
        _case("opt-1.3b next 8", "opt", "1.3b", 24, "next", 8, 8 * 1536, portion=0),
        # a full server: 64 requests of very different lengths
        _case("opt-1.3b next 64", "opt", "1.3b", 24, "next", 64, 64 * 1000 + 9, portion=0),
        # the headline prompt: 2,048 tokens in one step
        _case("opt-1.3b prompt 2048", "opt", "1.3b", 24, "generate", 1, 2047),
        # serving with portions: 63 requests decode beside 512 tokens of a new prompt, at the widest layers
        _case("opt-6.7b mixed", "opt", "6.7b", 8, "next", 63, 63 * 601, portion=512),
        # true 32-bit: three prompts of odd lengths
        _case("opt-1.3b fp32 prompts", "opt", "1.3b", 24, "generate", 3, 701, dtype="fp32"),
        # a long prompt through gated linear attention, latent attention and routed experts
        _case("zitupel-1.3b prompt 2048", "zitupel", "1.3b", 8, "generate", 1, 2011),
        # several prompts at once through the state-space recurrence, the delta rule and coupled window attention
        _case("zimorax-1.3b prompts", "zimorax", "1.3b", 8, "generate", 3, 2048),
        # a longer prompt in two portions through windows that keep the first tokens, and retention
        _case("gisedra-1.3b portions", "gisedra", "1.3b", 8, "generate", 1, 1777, portion=1024),
        # eight requests from prompt to answer
        _case("pupalix-1.3b generate 8", "pupalix", "1.3b", 8, "generate", 8, 901, new=16),
        # one user's short exchange on the smallest sizes
        _case("fiterax-125m generate 1", "fiterax", "125m", 8, "generate", 1, 33, new=24),
        # a busy server at the widest layers: prompts in portions beside decoding
        _case("fefozen-6.7b generate 24", "fefozen", "6.7b", 8, "generate", 24, 2999, new=8, portion=512),
    ]


def draw(rng):
    """One more case: any family, 125m to 2.7b layer sizes (6.7b too for short passes), 1 to 48 requests, 1 to about 2,000 tokens
    a request."""
    most = max(_cost(c) for c in listed())
    while True:
        family = rng.choice(FAMILIES)
        size = rng.choice(("125m", "1.3b", "1.3b", "2.7b", "6.7b"))
        kind = rng.choice(("next", "generate") if family == "opt" else ("generate",))
        dtype = "fp32" if rng.random() < 0.15 else "bf16"
        layers = rng.choice((4, 8))
        requests = int(round(math.exp(rng.uniform(0.0, math.log(48)))))
        if kind == "next":
            tokens = int(requests * math.exp(rng.uniform(math.log(16), math.log(1800))))
            new, portion = 0, rng.choice((0, 0, int(math.exp(rng.uniform(math.log(2), math.log(1024))))))
        else:
            tokens = int(math.exp(rng.uniform(math.log(2 * requests), math.log(4096))))
            tokens = max(requests, min(tokens, 1000 * requests + 900))
            new = rng.choice((0, 0, rng.randint(1, 16)))
            portion = rng.choice((512, 1024, BUDGET))
        case = _case("", family, size, layers, kind, requests, tokens, new, portion, dtype)
        if _cost(case) <= most and (dtype == "bf16" or tokens <= 1500):
            return case


# ------------------------------------------------------------------------------------------------- requests and their steps
def _lengths(case):
    """How many tokens of prompt or context each request has: ragged, at most 1,990 (the shortest position limit is 2,048)."""
    n, total = case["requests"], case["tokens"]
    rng = random.Random(f"{n} requests of {total} tokens")
    share = [rng.uniform(0.3, 1.7) for _ in range(n)] if n > 1 else [1.0]
    most = 2047 if n == 1 else 1990
    lens = [min(most, max(1, int(total * s / sum(share)))) for s in share]
    while sum(lens) < total and min(lens) < most:
        k = lens.index(min(lens))
        lens[k] += min(total - sum(lens), most - lens[k], max(1, total // (8 * n)))
    return lens


def _steps(case):
    """The steps of a "generate" pass: lists of (request, first position, tokens, whether the last row is wanted)."""
    lens = _lengths(case)
    at, steps = [0] * len(lens), []
    end = [n + case["new"] for n in lens]
    while any(a < e for a, e in zip(at, end)):
        room, step = BUDGET, []
        for r, n in enumerate(lens):
            if n <= at[r] < end[r]:
                step.append((r, at[r], 1, True))
                room -= 1
        for r, n in enumerate(lens):
            take = min(n - at[r], case["portion"], room) if at[r] < n else 0
            if take > 0:
                step.append((r, at[r], take, at[r] + take == n))
                room -= take
        for r, _a, n, _w in step:
            at[r] += n
        steps.append(step)
    return steps


def _hyper(case):
    key = "num_hidden_layers" if case["family"] == "opt" else "num_layers"
    return hyper_param_by_name(f"{case['family']}_{case['size']}", **{key: case["layers"]})


# ------------------------------------------------------------------------------------------------- weights and tokens
EMBED_NAMES = ("embed", "model.decoder.embed_tokens.weight")


def _weights(case, seed):
    """name -> tensor for every tensor that the model declares, in the types it keeps them in.  Matrices are N(0, 0.02) and gains
    1 + N(0, 0.1); time constants, gates and filters have the ranges they are trained from."""
    hp = _hyper(case)
    model = build_model(hp, DTYPES[case["dtype"]])
    specs = [s for s in model.tensor_specs() if not s.optional]
    g = torch.Generator(device="cuda").manual_seed(seed * 1009 + 17)
    normal = lambda shape, std: torch.empty(shape, device="cuda").normal_(0.0, std, generator=g)
    uniform = lambda shape, lo, hi: torch.empty(shape, device="cuda").uniform_(lo, hi, generator=g)
    w = {}
    for s in specs:
        if s.init == "gain":
            t = normal(s.shape, 0.1) + 1.0
        elif s.init == "mix":
            t = normal(s.shape, 0.1) + torch.eye(*s.shape, device="cuda")
        elif s.name.endswith("A_log"):
            t = uniform(s.shape, 1.0, 16.0).log()
        elif s.name.endswith("dt_bias"):
            t = uniform(s.shape, math.log(1e-3), math.log(0.1)).exp().expm1().log()
        elif s.name.endswith(".mix.f.b"):
            t = uniform(s.shape, 3.0, 6.0)
        elif s.name.endswith(".conv") or ".canon" in s.name:
            t = normal(s.shape, 0.5 if s.name.endswith(".conv") else 0.2)
        else:
            t = normal(s.shape, 0.02)
        w[s.name] = t
    _routers(w, case, g)
    for s in specs:
        keep = DTYPES[case["dtype"]] if s.kind in ("matrix", "table") else torch.float32
        w[s.name] = w[s.name].to(torch.bfloat16).to(keep)
    return model, w


def _routers(w, case, g):
    """Router rows are unit directions and every token's embedding holds two of them, the first the stronger.  The embedding's
    size is that of the branches that are added to it, where the model does not bring it to one itself."""
    routers = [n for n in w if n.endswith("mlp.router")]
    if not routers:
        return
    table = w["embed"]
    V, H = table.shape
    if case["family"] in ("pupalix", "fiterax"):
        size = 2.0 * H ** -0.5                                   # these multiply it by sqrt(H)
    else:
        size = 2.0
    table *= size / 0.02
    E = w[routers[0]].shape[0]
    dirs = torch.empty(E, H, device="cuda").normal_(0.0, 1.0, generator=g)
    dirs /= dirs.norm(dim=1, keepdim=True)
    first = torch.randint(0, E, (V,), device="cuda", generator=g)
    second = (first + torch.randint(1, E, (V,), device="cuda", generator=g)) % E
    table += (dirs[first] * 1.2 + dirs[second] * 0.8) * (size * H ** 0.5)
    for n in routers:
        perm = torch.randperm(E, device="cuda", generator=g)
        w[n] = dirs[perm] * 0.2 + w[n] * 0.05


def _tokens(case, seed, n, which):
    rng = torch.Generator().manual_seed(seed * 4099 + which)
    return (50272.0 ** torch.rand(n, generator=rng, dtype=torch.float64)).long().clamp_(0, 50271).tolist()


# ------------------------------------------------------------------------------------------------- the four functions
def _sequences(case, seed):
    """Every request's whole token sequence."""
    extra = 1 if case["kind"] == "next" else case["new"]
    seqs = [_tokens(case, seed, n + extra, r) for r, n in enumerate(_lengths(case))]
    if case["kind"] == "next" and case["portion"]:
        seqs.append(_tokens(case, seed, case["portion"], len(seqs)))
    return seqs


def prepare(case, seed):
    model, w = _weights(case, seed)
    model.bind(w)
    del w
    seqs = _sequences(case, seed)
    n = len(seqs)
    pages = sum(-(-(len(s) + 1) // PAGE) for s in seqs) + 8
    budget = BUDGET + n
    runner = ModelRunner(model, CacheParam(page_size=PAGE, num_pages=pages, max_seqs=n), "cuda:0", max_batched_tokens=budget)
    if case["kind"] == "next":
        fill, room = [], BUDGET
        for r, n_ctx in enumerate(_lengths(case)):
            runner.admit(r)
            if fill and n_ctx > room:
                runner.step(fill)
                fill, room = [], BUDGET
            fill.append(StepEntry(r, seqs[r][:n_ctx], []))
            room -= n_ctx
        runner.step(fill)
        entries = [StepEntry(r, seqs[r][-1:], [0]) for r in range(case["requests"])]
        if case["portion"]:
            runner.admit(case["requests"])
            entries.append(StepEntry(case["requests"], seqs[-1], [case["portion"] - 1]))
        state = {"runner": runner, "items": runner.prepare(entries)}
    else:
        steps, ends, done = [], [], set()
        for step in _steps(case):
            steps.append([StepEntry(r, seqs[r][a:a + m], [m - 1] if want else []) for r, a, m, want in step])
            ends.append([r for r, a, m, _w in step if a + m == len(seqs[r]) and r not in done])
            done.update(ends[-1])
        rows = sum(len(e.want) for s in steps for e in s)
        out = torch.empty((rows, model.vocab_size), dtype=torch.float32, device="cuda")
        state = {"runner": runner, "requests": n, "steps": steps, "ends": ends, "out": out}
    for _ in range(2):              # a server records its steps before the first request
        run(state)
    return state


def run(state):
    runner = state["runner"]
    if "items" in state:
        return runner.run(state["items"])
    out, at = state["out"], 0
    for r in range(state["requests"]):
        runner.admit(r)
    for entries, ends in zip(state["steps"], state["ends"]):
        logits = runner.step(entries)
        out[at:at + logits.shape[0]].copy_(logits)
        at += logits.shape[0]
        for r in ends:
            runner.finish(r)
    return out


def _parts(case):
    """(per layer: (dense matrix elements, elements of one expert, experts, a token's share of them, how often it runs, mixer)),
    head elements, width, whether a mixer's cache is shared by layer."""
    hp = _hyper(case)
    model = build_model(hp, DTYPES[case["dtype"]])
    runs = {}
    for e in model.schedule:
        runs[e.layer] = runs.get(e.layer, 0) + 1
    dense, expert, experts = {}, {}, {}
    for s in model.tensor_specs():
        m = re.match(r"(?:model\.decoder\.layers\.|l)(\d+)\.", s.name)
        if m is None or s.kind not in ("matrix",) or s.optional:
            continue
        i, size = int(m.group(1)), math.prod(s.shape)
        e = re.search(r"\.e(\d+)\.", s.name)
        if e is None:
            dense[i] = dense.get(i, 0) + size
        else:
            experts[i] = max(experts.get(i, 0), int(e.group(1)) + 1)
            expert[i] = expert.get(i, 0) + size
    layers = []
    for i in sorted(runs):
        if case["family"] == "opt":
            mixer = {"heads": hp.num_attention_heads, "kv_heads": hp.num_attention_heads,
                     "dim": hp.hidden_size // hp.num_attention_heads}
            kind, top = "attention", 0
        else:
            L = hp.layers[i]
            mixer, kind = L["mixer"], L["type"]
            top = (L.get("mlp") or {}).get("router", {}).get("top", 0)
        n = experts.get(i, 0)
        layers.append((dense.get(i, 0), expert.get(i, 0) / n if n else 0, n, top, runs[i], kind, mixer))
    width = hp.hidden_size if case["family"] == "opt" else hp.width
    return layers, 50272 * width, width


def work(case):
    """Weights once a step (an expert's only if a token is routed to it), the head's products of the wanted rows, cache entries that
    a query sees, recurrent states in and out, logits out; two operations a weight and token, four a visible pair and channel."""
    elem = 2 if case["dtype"] == "bf16" else 4
    layers, head, width = _parts(case)
    if case["kind"] == "next":
        step = [(r, n, 1, True) for r, n in enumerate(_lengths(case))]
        if case["portion"]:
            step.append((len(step), 0, case["portion"], True))
        steps = [step]
    else:
        steps = _steps(case)
    nbytes = flops = 0.0
    for step in steps:
        T = sum(n for _r, _a, n, _w in step)
        R = sum(1 for _r, _a, _n, w in step if w)
        nbytes += T * width * elem + R * 50272 * 4 + (head * elem if R else 0)
        flops += 2.0 * R * head
        for dense, expert, experts, top, runs, kind, mixer in layers:
            met = experts * (1.0 - (1.0 - top / experts) ** T) if experts else 0.0
            nbytes += (dense + expert * met) * elem
            flops += 2.0 * T * (dense + expert * min(top, experts)) * runs
            branches = [("attention", mixer["left"]), ("retention", mixer["right"])] if kind == "parallel" else [(kind, mixer)]
            for k, m in branches:
                for _r, a, n, _w in step:
                    if k in ("attention", "latent_attention", "latent_attention_2"):
                        window = (m.get("mask") or {}).get("size") or 10 ** 9
                        pairs = sum(min(p + 1, window) for p in range(a, a + n)) if n < 64 else n * (min(a + 0.5 * n, window))
                        seen = min(a + n, window + n)
                        if k == "attention":
                            entry = m["kv_heads"] * (m["dim"] + m.get("vdim", m["dim"]))
                        else:
                            entry = m["kv_rank"] + m.get("rot_dim", 0)
                        nbytes += seen * entry * elem * runs
                        flops += 2.0 * pairs * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m.get("vdim", m["dim"])) * runs
                    else:
                        state = m["heads"] * m.get("dim", m.get("state", 0)) * m["vdim"]
                        nbytes += 8.0 * state * runs
                        flops += 4.0 * n * state * runs
    return {"bytes": nbytes, "flops": flops}


def _cost(case):
    w = work(case)
    return w["bytes"] / 6e12 + w["flops"] / (1e15 if case["dtype"] == "bf16" else 1e14)


def tolerance(case):
    """About four times the measured distance of the logits from ``exact`` (relative, 2-norm).  bfloat16 storage between layers: some
    per mille, by how much of a model's logits its layers make up beside the token's own embedding.  float32: 1e-6 to 4e-6."""
    if case["dtype"] == "fp32":
        return {"rel": 1.5e-5, "max": 1e-3}
    rel = {"opt": 0.02, "zitupel": 0.02, "zimorax": 0.03, "gisedra": 0.01, "pupalix": 0.005, "fiterax": 0.008, "fefozen": 0.002}
    return {"rel": rel[case["family"]], "max": 0.3}


def exact(case, seed):
    """The same logits in float64, every sequence whole, from the formulas of the architectures."""
    _model, w = _weights(case, seed)
    cfg = _hyper(case).to_config_dict()
    seqs = _sequences(case, seed)
    if case["kind"] == "next":
        wanted = [(r, len(s) - 1) for r, s in enumerate(seqs)]
    else:
        wanted = [(r, a + n - 1) for step in _steps(case) for r, a, n, want in step if want]
    out = torch.empty((len(wanted), 50272), dtype=torch.float64, device="cuda")
    for r, seq in enumerate(seqs):
        at = [i for i, (q, _p) in enumerate(wanted) if q == r]
        rows = torch.tensor([wanted[i][1] for i in at], device="cuda")
        out[at] = _PLAIN[case["family"]](cfg, _Plain(w), torch.tensor(seq, device="cuda"), rows)
    return out


# ------------------------------------------------------------------------------------------------- the formulas in float64
class _Plain:
    """Weights by name, in float64 when asked for."""

    def __init__(self, w, prefix=""):
        self.w, self.prefix = w, prefix

    def __getitem__(self, name):
        return self.w[self.prefix + name].double()

    def __contains__(self, name):
        return self.prefix + name in self.w

    def under(self, prefix):
        return _Plain(self.w, self.prefix + prefix)


def _ln(x, gain, bias, eps):
    d = x - x.mean(-1, keepdim=True)
    y = d / torch.sqrt(d.square().mean(-1, keepdim=True) + eps) * gain
    return y if bias is None else y + bias


def _rms(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))


def _gelu_tanh(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _filter(x, w, bias=None):
    """A causal filter over time; the last column of w meets the row itself."""
    n = w.shape[1]
    y = torch.zeros_like(x)
    for j in range(n):
        back = n - 1 - j
        if back < x.shape[0]:
            y[back:] += w[:, j] * x[:x.shape[0] - back]
    return y if bias is None else y + bias


def _frequencies(rot):
    dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
    i = torch.arange(dims // 2, device="cuda", dtype=torch.float64)
    f = base ** (-2 * i / dims)
    if not sc:
        return f, 1.0
    if "low" in sc:
        turns = sc["original"] * f / (2 * math.pi)                 # wavelengths within the original context
        s = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
        return (1 - s) * f / sc["factor"] + s * f, 1.0
    border = lambda t: dims * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(base))
    lo, hi = max(math.floor(border(sc["fast"])), 0), min(math.ceil(border(sc["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def _turn(x, rot, pairs):
    """x [T, heads, n]: the first ``dims`` coordinates turn by position; ``pairs``: neighbours turn together, else halves."""
    if not rot:
        return x
    dims = rot["dims"]
    f, mult = _frequencies(rot)
    a = torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None] * f
    c, s = (a.cos() * mult)[:, None], (a.sin() * mult)[:, None]
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if pairs else (x[..., :dims // 2], x[..., dims // 2:dims])
    y = x.clone()
    if pairs:
        y[..., 0:dims:2], y[..., 1:dims:2] = u * c - v * s, v * c + u * s
    else:
        y[..., :dims // 2], y[..., dims // 2:dims] = u * c - v * s, v * c + u * s
    return y


def _attend(q, k, v, scale, size=0, keep=0, chunk=0, cap=0.0, mix=None, sink=None):
    """q [T, heads, d], k and v [T, kv heads, .] -> [T, heads, dv].  ``sink``: one more logit a head in the denominator."""
    T, H, _ = q.shape
    rep = H // k.shape[1]
    k, v = k.repeat_interleave(rep, 1).transpose(0, 1).contiguous(), v.repeat_interleave(rep, 1).transpose(0, 1).contiguous()
    i, j = torch.arange(T, device="cuda")[:, None], torch.arange(T, device="cuda")[None]
    seen = j <= i
    if size:
        seen = seen & ((i - j < size) | (j < keep))
    if chunk:
        seen = seen & (i // chunk == j // chunk)
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device="cuda")
    for a in range(0, T, 512):                                     # rows at a time
        b = min(T, a + 512)
        s = q[a:b].transpose(0, 1).contiguous() @ k.transpose(1, 2).contiguous() * scale
        if mix is not None:
            s = (mix @ s.reshape(H, -1)).reshape(s.shape)
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~seen[None, a:b], -math.inf)
        top = s.amax(-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink[:, None, None])
        p = torch.exp(s - top)
        total = p.sum(-1, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sink[:, None, None] - top)
        out[a:b] = (p / total @ v).transpose(0, 1)
    return out


def _walk(q, k, v, decay, delta=None):
    """S <- decay S + k v^T, o = S^T q, token by token; decay [T, heads] or [T, heads, d].  ``delta`` [T, heads]: the delta rule's
    strength, S <- decay S, then S += k (delta (v - S^T k))^T."""
    T, H, d = q.shape
    S = torch.zeros(H, d, v.shape[2], dtype=q.dtype, device="cuda")
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device="cuda")
    decay = decay.reshape(T, H, -1, 1)
    for t in range(T):
        S = decay[t] * S
        u = v[t] if delta is None else delta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S += k[t][:, :, None] * u[:, None, :]
        torch.sum(S * q[t][:, :, None], 1, out=out[t])
    return out


def _experts(h, scores, weights, top, unit):
    """sum over the ``top`` best by ``scores`` [T, E] of unit(e, rows, weights of these rows)."""
    out = torch.zeros_like(h)
    best = torch.topk(scores, top, dim=1).indices
    for e in range(scores.shape[1]):
        rows = (best == e).any(1).nonzero()[:, 0]
        if rows.numel():
            out[rows] += unit(e, h[rows], weights(rows, e, best))
    return out


def _gated_expert(w, limit=None):
    def unit(x, e):
        g, u = x @ w[f"e{e}.gate"].T, x @ w[f"e{e}.up"].T
        if limit is None:
            return (_silu(g) * u) @ w[f"e{e}.down"].T
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[f"e{e}.down"].T
    return unit


def _order(cfg):
    """[(layer, number of the pass that starts here or None)]."""
    n, loop = len(cfg["layers"]), cfg.get("loop")
    if not loop:
        return [(i, None) for i in range(n)]
    a, b = loop["start"], loop["stop"]
    passes = [(i, t if i == a else None) for t in range(loop["times"]) for i in range(a, b)]
    return [(i, None) for i in range(a)] + passes + [(i, None) for i in range(b, n)]


def _opt(cfg, w, tokens, rows):
    T, H = tokens.shape[0], cfg["hidden_size"]
    heads = cfg["num_attention_heads"]
    w = w.under("model.decoder.")
    norm = lambda x, name: _ln(x, w[name + ".weight"], w[name + ".bias"], 1e-5)
    x = w["embed_tokens.weight"][tokens] + w["embed_positions.weight"][2:2 + T]
    for i in range(cfg["num_hidden_layers"]):
        p = w.under(f"layers.{i}.")
        lin = lambda y, n: y @ p[n + ".weight"].T + p[n + ".bias"]
        h = norm(x, f"layers.{i}.self_attn_layer_norm")
        q, k, v = (lin(h, f"self_attn.{n}_proj").view(T, heads, -1) for n in "qkv")
        x = x + lin(_attend(q, k, v, (H // heads) ** -0.5).reshape(T, H), "self_attn.out_proj")
        x = x + lin(torch.relu(lin(norm(x, f"layers.{i}.final_layer_norm"), "fc1")), "fc2")
    return norm(x[rows], "final_layer_norm") @ w["embed_tokens.weight"].T


def _zitupel(cfg, w, tokens, rows):
    eps, mult, T = cfg["norm"]["eps"], cfg["residual_mult"], tokens.shape[0]
    x = _rms(w["embed"][tokens], eps) * w["embed.norm"]
    latents = {}
    for i, L in enumerate(cfg["layers"]):
        p, m, mlp = w.under(f"l{i}.mix."), L["mixer"], L["mlp"]
        h = _rms(x, eps) * w[f"l{i}.norm1"]
        if cfg.get("canon"):
            h = h + _filter(h, w[f"l{i}.canon1"])
        heads = lambda n, src: (src @ p[n].T).view(T, m["heads"], -1)
        if L["type"] == "gla":
            decay = torch.sigmoid(h @ p["a1"].T @ p["a2"].T + p["a2.b"]) ** (1.0 / m["tau"])
            o = _walk(heads("q", h) * m["dim"] ** -0.5, heads("k", h), heads("v", h), decay.view(T, m["heads"], -1))
            y = (_rms(o, eps) * p["norm"]).reshape(T, -1) * _silu(h @ p["g"].T)
        else:
            src = m.get("kv_from")
            latents[i] = _rms(h @ p["dkv"].T, eps) * p["dkv.norm"] if src is None else latents[src]
            y = _attend(heads("q", h), heads("uk", latents[i]), heads("uv", latents[i]), m["scale"]).reshape(T, -1)
        x = x + mult * (y @ p["o"].T)
        h, p = _rms(x, eps) * w[f"l{i}.norm2"], w.under(f"l{i}.mlp.")
        if mlp["kind"] == "dense":
            x = x + mult * (_gelu(h @ p["up"].T) @ p["down"].T)
        else:
            s = torch.sigmoid(h @ p["router"].T)
            unit = _gated_expert(p, mlp["expert"]["limit"])
            x = x + mult * _experts(h, s, lambda r, e, _b: s[r, e:e + 1], mlp["router"]["top"], lambda e, y, g: unit(g * y, e))
    return _rms(x[rows], eps) * w["final.norm"] @ w["head"].T


def _delta_rule(h, p, m, eps):
    T, rep = h.shape[0], m["heads"] // m["kv_heads"]
    q, k, v = (_silu(_filter(h @ p[n].T, p[n + ".conv"])) for n in "qkv")
    unit = lambda y: y / torch.sqrt(y.square().sum(-1, keepdim=True) + 1e-6)
    q, k = (unit(y.view(T, m["kv_heads"], -1)).repeat_interleave(rep, 1) for y in (q, k))
    decay = torch.exp(-torch.exp(p["A_log"]) * torch.nn.functional.softplus(h @ p["a"].T + p["dt_bias"]))
    o = _walk(q * m["dim"] ** -0.5, k, v.view(T, m["heads"], -1), decay, torch.sigmoid(h @ p["b"].T))
    return ((_rms(o, eps) * p["norm"]).reshape(T, -1) * _silu(h @ p["g"].T)) @ p["o"].T


def _zimorax(cfg, w, tokens, rows):
    eps, T = cfg["norm"]["eps"], tokens.shape[0]
    first = x = w["embed"][tokens]
    for i, pass_no in _order(cfg):
        if pass_no is not None:
            x = torch.cat([x, first], -1) @ w["loop.in"].T + w["loop.step"][pass_no]
        L, p, m = cfg["layers"][i], w.under(f"l{i}.mix."), cfg["layers"][i]["mixer"]
        h = _ln(x, w[f"l{i}.norm1"], None, eps)
        if L["type"] == "attention":
            q, k, v = ((h @ p[n].T + p[n + ".b"]).view(T, -1, m["vdim"] if n == "v" else m["dim"]) for n in "qkv")
            sink = torch.zeros(m["heads"], dtype=x.dtype, device="cuda")
            y = _attend(_turn(q, m["rot"], False), _turn(k, m["rot"], False), _rms(v, eps), m["scale"], m["mask"]["size"],
                        mix=p["talk"], sink=sink).reshape(T, -1) @ p["o"].T
        elif L["type"] == "mamba2":
            inner, bc = m["heads"] * m["vdim"], m["groups"] * m["state"]
            z, u, dt = (h @ p["in"].T).split([inner, inner + 2 * bc, m["heads"]], -1)
            u = _silu(_filter(u, p["conv"], p["conv.b"]))
            rep = m["heads"] // m["groups"]
            v = u[:, :inner].reshape(T, m["heads"], -1)
            b, c = (y.reshape(T, m["groups"], -1).repeat_interleave(rep, 1) for y in (u[:, inner:inner + bc], u[:, inner + bc:]))
            dt = torch.nn.functional.softplus(dt + p["dt_bias"])
            y = _walk(c, b * dt[:, :, None], v, torch.exp(-torch.exp(p["A_log"]) * dt)) + p["D"][:, None] * v
            y = _rms((y.reshape(T, inner) * _silu(z)).view(T, m["norm_groups"], -1), eps).reshape(T, inner) * p["norm"] @ p["o"].T
        else:
            y = _delta_rule(h, p, m, eps)
        x = x + w[f"l{i}.ls1"] * y
        h, p = _ln(x, w[f"l{i}.norm2"], None, eps), w.under(f"l{i}.mlp.")
        x = x + w[f"l{i}.ls2"] * (torch.relu(h @ p["up"].T + p["up.b"]).square() @ p["down"].T + p["down.b"])
    return _ln(x[rows], w["final.norm"], None, eps) @ w["head"].T


def _latent(h, p, m, eps, size=0):
    """Keys and values from one normed latent; a turned key part shared by the heads."""
    T, d, R = h.shape[0], m["dim"], m["kv_rank"]
    q, down = (h @ p["q"].T).view(T, m["heads"], -1), h @ p["dkv"].T
    c = _rms(down[:, :R], eps) * p["dkv.norm"]
    k_turned = _turn(down[:, None, R:], m["rot"], True).expand(-1, m["heads"], -1)
    q = torch.cat([q[..., :d], _turn(q[..., d:], m["rot"], True)], -1)
    k = torch.cat([(c @ p["uk"].T).view(T, m["heads"], d), k_turned], -1)
    return _attend(q, k, (c @ p["uv"].T).view(T, m["heads"], -1), m["scale"], size).reshape(T, -1) @ p["o"].T


def _gisedra(cfg, w, tokens, rows):
    eps, T = cfg["norm"]["eps"], tokens.shape[0]
    norm = lambda y, n: torch.tanh(w[n + ".alpha"] * y) * w[n] + w[n + ".b"]
    first = x = w["embed"][tokens]
    for i, pass_no in _order(cfg):
        if pass_no is not None:
            x = x + (first if pass_no > 0 else 0) + w["loop.step"][pass_no]
        L, m, mlp = cfg["layers"][i], cfg["layers"][i]["mixer"], cfg["layers"][i]["mlp"]
        h = norm(x, f"l{i}.norm1")
        if L["type"] == "parallel":
            p, a = w.under(f"l{i}.mix.left."), m["left"]
            q, k, v = (_filter(h @ p[n].T, p[n + ".conv"]).view(T, -1, a["vdim"] if n == "v" else a["dim"]) for n in "qkv")
            o = _attend(_turn(q, a["rot"], False), _turn(k, a["rot"], False), v, a["scale"], a["mask"]["size"],
                        a["mask"]["keep_first"])
            y = m["left_scale"] * ((o.reshape(T, -1) * torch.sigmoid(h @ p["g"].T)) @ p["o"].T)
            p, a = w.under(f"l{i}.mix.right."), m["right"]
            q, k, v = ((h @ p[n].T).view(T, a["heads"], -1) for n in "qkv")
            decay = torch.tensor(a["decay"], dtype=x.dtype, device="cuda").expand(T, -1)
            o = _rms(_walk(q, k * a["dim"] ** -0.5, v, decay), eps).reshape(T, -1) * _silu(h @ p["g"].T)
            y = y + m["right_scale"] * (o @ p["o"].T)
        else:
            y = _latent(h, w.under(f"l{i}.mix."), m, eps, m["mask"]["size"])
        x = x + norm(y, f"l{i}.norm1b")
        h, p = norm(x, f"l{i}.norm2"), w.under(f"l{i}.mlp.")
        z = h @ p["router"].T + p["router.b"]
        unit = _gated_expert(p)
        share = lambda r, e, best: torch.exp(z[r, e:e + 1] - torch.logsumexp(z[r].gather(1, best[r]), 1, True))
        x = x + norm(_experts(h, z, share, mlp["router"]["top"], lambda e, y, g: g * unit(y, e)), f"l{i}.norm2b")
        d, p = cfg["token_side"]["dim"], w.under(f"l{i}.side.")
        side = (_gelu_tanh(x @ p["gate"].T) * w["side.embed"][tokens][:, i * d:(i + 1) * d]) @ p["proj"].T
        x = x + _rms(side, eps) * p["norm"]
    return norm(x[rows], "final.norm") @ w["head"].T


def _pupalix(cfg, w, tokens, rows):
    eps, T, emb = cfg["norm"]["eps"], tokens.shape[0], cfg["embedding"]
    rule = emb["bigram"]
    pair = torch.full((T,), rule["buckets"], device="cuda")
    pair[1:] = (tokens[:-1] * rule["mul_prev"] + tokens[1:] * rule["mul_cur"]) % rule["buckets"]
    xs = (w["embed"][tokens] * emb["scale"] + w["bigram"][pair]).expand(cfg["streams"], -1, -1)

    def around(xs, hc, norm, sublayer):
        S = xs.shape[0]
        y = sublayer(_rms((hc["in"] @ xs.reshape(S, -1)).view(T, -1), eps) * norm)
        return (hc["mix"].T @ xs.reshape(S, -1)).view(xs.shape) + hc["out"][:, None, None] * y

    def mixer(h, L, p):
        m = L["mixer"]
        if L["type"] == "latent_attention":
            return _latent(h, p, m, eps)
        if L["type"] == "attention":
            q, k = h @ p["q"].T, h @ p["k"].T
            split = lambda y: y.view(T, -1, m["dim"])
            return _attend(split(_rms(q, eps) * p["q.norm"]), split(_rms(k, eps) * p["k.norm"]), split(k), m["scale"],
                           chunk=m["mask"]["size"], cap=m["softcap"]).reshape(T, -1) @ p["o"].T
        q, k, v = (_silu(h @ p[n].T).view(T, m["heads"], -1) for n in "qkv")
        o = _walk(q, k, v, torch.tensor(m["decay"], dtype=h.dtype, device="cuda").expand(T, -1)).reshape(T, -1)
        return (_rms(o, eps) * p["norm"] * torch.sigmoid(h @ p["g"].T)) @ p["o"].T

    def feed_forward(h, mlp, p):
        if mlp["kind"] == "dense":
            return (_gelu_tanh(h @ p["gate"].T) * (h @ p["up"].T)) @ p["down"].T
        r = mlp["router"]
        s = torch.softmax(h @ p["router"].T, -1)
        groups = s.view(T, r["groups"]["count"], -1)
        kept = torch.zeros(groups.shape[:2], dtype=torch.bool, device="cuda")
        kept.scatter_(1, torch.topk(groups.amax(2), r["groups"]["keep"], dim=1).indices, True)
        allowed = groups.masked_fill(~kept[:, :, None], -1.0).view(T, -1)
        unit = _gated_expert(p)
        return _experts(h, allowed, lambda q, e, _b: s[q, e:e + 1], r["top"], lambda e, y, g: g * unit(y, e))

    for i, _pass in _order(cfg):
        L = cfg["layers"][i]
        xs = around(xs, w.under(f"l{i}.hc1."), w[f"l{i}.norm1"], lambda h: mixer(h, L, w.under(f"l{i}.mix.")))
        xs = around(xs, w.under(f"l{i}.hc2."), w[f"l{i}.norm2"], lambda h: feed_forward(h, L["mlp"], w.under(f"l{i}.mlp.")))
    z = _rms(xs.sum(0)[rows], eps) * w["final.norm"] @ w["embed"].T * cfg["logit_scale"]
    return cfg["logit_softcap"] * torch.tanh(z / cfg["logit_softcap"])


def _fiterax(cfg, w, tokens, rows):
    eps, T, groups = cfg["norm"]["eps"], tokens.shape[0], cfg["norm"]["groups"]
    norm = lambda y, n: _rms(y.reshape(y.shape[0], groups, -1), eps).reshape(y.shape) * w[n]
    x = w["embed"][tokens] * cfg["embedding"]["scale"]

    def read(i, side):
        h = norm(x, f"l{i}.norm{side}")
        return h + _filter(h, w[f"l{i}.canon{side}"]) if cfg.get("canon") else h

    def memory(h, p, m):
        q, k, v = ((h @ p[n].T).view(T, m["heads"], -1) for n in "qkv")
        q = q * m["dim"] ** -0.5
        squash = lambda n: m["gate_cap"] * torch.tanh((h @ p[n].T + p[n + ".b"]) / m["gate_cap"])
        i, f = squash("i"), torch.nn.functional.logsigmoid(squash("f"))
        # the running maximum only keeps numbers small: with the memory relative to it, every step's factors follow at once
        total = torch.cumsum(f, 0)
        top = torch.maximum(torch.cummax(i - total, 0).values, torch.zeros((), dtype=h.dtype, device="cuda"))
        before = torch.cat([torch.zeros_like(top[:1]), top[:-1]])
        decay, add = torch.exp(before - top), torch.exp(i - total - top)
        vn = torch.cat([v, torch.ones_like(v[..., :1])], -1)        # the normaliser is one more value channel
        o = _walk(q, k * add[:, :, None], vn, decay)
        o = o[..., :-1] / (torch.maximum(o[..., -1:].abs(), torch.exp(-total - top)[..., None]) + 1e-6)
        return (_rms(o, eps).reshape(T, -1) * p["norm"] * torch.sigmoid(h @ p["g"].T)) @ p["o"].T

    for i, L in enumerate(cfg["layers"]):
        m, mlp, p = L["mixer"], L["mlp"], w.under(f"l{i}.mix.")
        h = read(i, 1)
        if L["type"] == "attention":
            q, k, v = ((h @ p[n].T + p[n + ".b"]).view(T, -1, m["vdim"] if n == "v" else m["dim"]) for n in "qkv")
            q = _rms(_turn(q, m["rot"], False), eps) * p["temp"][:, None]
            o = _attend(q, _rms(_turn(k, m["rot"], False), eps), v, m["scale"], cap=m["softcap"])
            y = (o * torch.sigmoid(h @ p["g"].T)[:, :, None]).reshape(T, -1) @ p["o"].T + p["o.b"]
        else:
            y = memory(h, p, m)
        h, p = read(i, 2), w.under(f"l{i}.mlp.")
        s = torch.sigmoid(h @ p["router"].T)
        share = lambda r, e, best: s[r, e:e + 1] / (s[r].gather(1, best[r]).sum(1, True) + 1e-20) * mlp["router"]["scale"]
        unit = lambda e, y, g: g * (_gelu(y @ p[f"e{e}.up"].T) @ p[f"e{e}.down"].T)
        x = x + cfg["residual_mult"] * (y + _experts(h, s + p["correction"], share, mlp["router"]["top"], unit))
    return norm(x[rows], "final.norm") @ w["head"].T


def _fefozen(cfg, w, tokens, rows):
    eps, T = cfg["norm"]["eps"], tokens.shape[0]
    norm = lambda y, n: _rms(y, eps) * (1 + w[n])
    x, cached = w["embed"][tokens], {}
    for i, L in enumerate(cfg["layers"]):
        m, mlp, p = L["mixer"], L["mlp"], w.under(f"l{i}.mix.")
        h = norm(x, f"l{i}.norm1")
        if L["type"] == "delta":
            y = _delta_rule(h, p, m, eps)
        else:
            pairs, src, d = L["type"] == "latent_attention", m.get("kv_from"), m["dim"]
            if src is None:
                raw = h @ p["dkv"].T
                cached[i] = (_rms(raw[:, :m["kv_rank"]], eps) * p["dkv.norm"], _turn(raw[:, None, m["kv_rank"]:], m["rot"], pairs))
            c, k_turned = cached[i if src is None else src]
            q = ((_rms(h @ p["dq"].T, eps) * p["dq.norm"]) @ p["uq"].T).view(T, m["heads"], -1)
            q = torch.cat([q[..., :d], _turn(q[..., d:], m["rot"], pairs)], -1)
            k = torch.cat([(c @ p["uk"].T).view(T, m["heads"], d), k_turned.expand(-1, m["heads"], -1)], -1)
            o = _attend(q, k, (c @ p["uv"].T).view(T, m["heads"], -1), m["scale"], sink=p["sink"] if pairs else None)
            y = (o.reshape(T, -1) * torch.sigmoid(h @ p["g"].T)) @ p["o"].T
        x = x + norm(y, f"l{i}.norm1b")
        h, p = norm(x, f"l{i}.norm2"), w.under(f"l{i}.mlp.")
        if mlp["kind"] == "dense":
            y = _gelu_tanh(h @ p["up"].T) @ p["down"].T
        else:
            s, n = torch.softmax(h @ p["router"].T, -1), mlp["router"]["experts"]
            unit = _gated_expert(p, mlp["expert"]["limit"])
            y = _experts(h, s + p["correction"], lambda r, e, _b: s[r, e:e + 1], mlp["router"]["top"],
                         lambda e, y, g: g * (unit(y, e) if e < n else y))
        x = x + norm(y, f"l{i}.norm2b")
    return norm(x[rows], "final.norm") @ w["embed"].T


_PLAIN = {"opt": _opt, "zitupel": _zitupel, "zimorax": _zimorax, "gisedra": _gisedra, "pupalix": _pupalix, "fiterax": _fiterax,
          "fefozen": _fefozen}
