"""Latent attention with entries above 128 in bfloat16, whose prompts go through the tiles made for a latent cache: the mixer alone (all keys,
windows, chunks; queries turned inside the tiles, and outside them beside single tokens or where the kernel cannot) and whole models, in
one step, in portions beside decoded tokens, recorded and not."""
import pytest
import torch

import plain_gisedra as plain
import tiny_gisedra as tiny
from test_parts_gpu import ctx_for
from test_zimorax_gpu import DEV, F64, check, make_runner, run_schedule

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _mixer(rank, rot, window, heads=4, dim=24, vdim=16, H=64):
    """The part, and its weights in float64 under the plain implementation's names (``m.q`` ...)."""
    from swifttransformer_amd.parts import PartSpec, build_part
    from swifttransformer_amd.weights import random_tensors
    spec = PartSpec("latent_attention", {"num_heads": heads, "key_dim": dim, "value_dim": vdim, "rank": rank, "scale": 0.4, "eps": 1e-5,
                                         "rot_dim": rot, "rot_base": 300.0, "window": window},
                    {"q": "m.q", "down": "m.dkv", "down_norm": "m.dkv.norm", "up_k": "m.uk", "up_v": "m.uv", "out": "m.o"})
    part = build_part("mixer", spec, H, BF16)
    t = random_tensors(part.tensor_specs(), rank + rot, BF16, DEV)
    for k in t:                        # scores far from even
        if not k.endswith("norm"):
            t[k] = (t[k] * 6.0).contiguous()
    part.bind(t)
    c = {"heads": heads, "dim": dim, "rot_dim": rot, "vdim": vdim, "kv_rank": rank, "scale": 0.4,
         "rot": {"dims": rot, "base": 300.0}, "mask": {"size": window}}
    return part, {k: v.to(F64).cpu() for k, v in t.items()}, c


def _visible(T, window):
    """Keys j of row i: all before it, the last ``window`` (> 0), or its chunk of -window (< 0)."""
    i, j = torch.arange(T)[:, None], torch.arange(T)[None, :]
    return (j <= i) & (i - j < window if window > 0 else j >= i - i % -window if window < 0 else j >= 0)


@pytest.mark.parametrize("rank,rot", [(128, 32), (132, 12), (160, 0), (240, 16)])          # 132: the tiles cannot turn these queries
@pytest.mark.parametrize("window", [0, 50, -48])
def test_large_entries_in_the_mixer(monkeypatch, rank, rot, window):
    from swifttransformer_amd.engine.batch import StepItem
    from swifttransformer_amd.ops import kernels as K
    from swifttransformer_amd.cache.device import CacheView
    part, w, c = _mixer(rank, rot, window)
    monkeypatch.setattr(plain, "visible", _visible)
    if rot == 0:
        monkeypatch.setattr(plain, "rotary_frequencies", lambda *a: [])
        monkeypatch.setattr(plain, "rotate", lambda x, *a: x)
    inside = []
    tiles = K.latent_tiles
    monkeypatch.setattr(K, "latent_tiles", lambda *a: (inside.append(a[8].freq is not None), tiles(*a)))
    n, ps = 460, 16
    x = {s: torch.randn(n, 64, generator=torch.Generator().manual_seed(s)).to(BF16) for s in (0, 1)}
    res = {s: torch.randn(n, 64, generator=torch.Generator().manual_seed(7 + s)) for s in (0, 1)}
    ref = {s: res[s].to(F64) + plain.latent_attention(x[s].to(F64), w, "m", c, 1e-5) for s in (0, 1)}
    pool = torch.full((64, 1, ps, part.entry), float("nan"), dtype=BF16, device=DEV)
    cache = CacheView(0, 0, k=pool, v=pool)
    order = torch.randperm(64, generator=torch.Generator().manual_seed(3)).tolist()
    pages = {0: order[:29], 1: order[29:58]}
    done, expected = {0: 0, 1: 0}, []
    least = (0 if part.entry <= 160 else 96) if rot and rank % 8 == 0 else None, 384 if part.entry <= 144 else 256
    # alone, few keys and many; beside the other's portion; single tokens beside a portion; single tokens alone; the rest
    for step in ([(0, 70)], [(0, 300)], [(1, 380), (0, 9)], [(0, 1), (1, 33)], [(1, 1), (0, 40)], [(0, 1), (1, 1)], [(0, 39), (1, 45)]):
        items = [StepItem(s, done[s], list(range(m)), [], {0: pages[s]}) for s, m in step]
        ctx = ctx_for(items, page_size=ps, max_pages=32, parts=[part])
        part_of = lambda v: torch.cat([v[s][done[s]:done[s] + m] for s, m in step])
        out = part.forward(part_of(x).to(DEV), part_of(res).to(DEV), ctx, cache)
        check(out, part_of(ref).numpy(), BF16, f"rank {rank} rot {rot} window {window} step {step}")
        for s, m in step:
            done[s] += m
        long = [done[s] if window == 0 else min(done[s], window + 64) for s, m in step if m >= 8]
        turned = least[0] is not None and all(m >= 8 for _, m in step)
        if long and window >= 0 and max(long) >= least[0 if turned else 1]:
            expected.append(turned)
    assert inside == expected


def test_a_plan_of_other_tiles_is_not_read_as_one_of_64_rows():
    from swifttransformer_amd.engine.batch import StepItem
    from swifttransformer_amd.ops import kernels as K
    from swifttransformer_amd.parts.attention import plan_tiles
    from swifttransformer_amd.cache.device import CacheView
    from swifttransformer_amd.parts.base import StepPlan
    part, _w, _c = _mixer(128, 32, 0)
    items = [StepItem(0, 0, list(range(130)), [], {0: list(range(9))})]
    ctx = ctx_for(items, page_size=16, parts=[part])
    plan = plan_tiles(items, 8, 128)
    plan.host["latent_tiles"] = 1
    arrays = {k: torch.from_numpy(v).to(DEV) for k, v in plan.arrays.items()}
    ctx.plans[part.plan_key()] = StepPlan(arrays, plan.host)
    pool = torch.zeros((9, 1, 16, part.entry), dtype=BF16, device=DEV)
    with pytest.raises(K.KernelError, match="128 rows"):
        part.forward(torch.randn(130, 64, device=DEV).to(BF16), torch.zeros(130, 64, device=DEV), ctx, CacheView(0, 0, k=pool, v=pool))


CONFIGS = {
    "rank 128": [tiny._with(tiny._latent(4, 24, 32, 16, 128, 0.3, window=70), tiny._moe(4, 2, 24)),
                 tiny._with(tiny._latent(4, 24, 32, 16, 128, 0.3), None)],
    "rank 132": [tiny._with(tiny._latent(3, 16, 12, 20, 132, 0.35), None)],
    "rank 240": [tiny._with(tiny._latent(2, 32, 16, 24, 240, 0.25, window=40), None)],
}


@pytest.mark.parametrize("recording", [0, 1, 2])
@pytest.mark.parametrize("name", list(CONFIGS))
def test_models_with_large_entries_against_the_plain_one(tmp_path, monkeypatch, name, recording):
    from swifttransformer_amd.ops import kernels as K
    cfg = {"architecture": "Gisedra", "vocab": 97, "width": 64, "max_positions": 512, "norm": {"eps": 1e-6}, "layers": CONFIGS[name]}
    folder = tiny.write_folder(cfg, str(tmp_path / "m"), 5)
    cfg, w = plain.load_folder(folder)
    seqs = {r: tiny.prompt(450, 97, i) for i, r in enumerate("ab")}
    refs = {r: plain.logits(cfg, w, s).numpy() for r, s in seqs.items()}
    calls = []
    tiles = K.latent_tiles
    monkeypatch.setattr(K, "latent_tiles", lambda *a: (calls.append(1), tiles(*a)))
    runner = make_runner(folder, "bfloat16", 16, 60, record_after=recording, max_seqs=2)
    what = f"{name} recording {recording}"
    for _ in range(2):                                # the second time on pages used before, and from recordings
        run_schedule(runner, seqs, refs, [[("a", 225)], [("a", 225)], [("b", 225)], [("b", 225)]], "bfloat16", what + " alone")
        run_schedule(runner, seqs, refs, [[("a", 60)], [("a", 1), ("b", 230)], [("b", 1), ("a", 240)], [("a", 1), ("b", 190)], [("a", 1), ("b", 1)],
                                          [("a", 147), ("b", 28)]], "bfloat16", what + " portions beside decoded tokens")
    assert calls
    if recording == 1:
        assert runner.graph_replays == runner.steps_run, "a step ran unrecorded"
