"""Window attention of prompts in tiles on the matrix cores, against float64: tiles with a last short one, single rows beside a
portion, portions that start behind the window, windows that are no multiple of a block and keep the first tokens, every key in one
block, heads alone, in fours and mixed (up to 16 and up to 32 of them), sizes up to the largest, rows of no item."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


@pytest.mark.parametrize("lens,starts,H,G,dk,dv,window,keep,sink,mixed", [
    ((128,), (0,), 4, 1, 64, 64, 0, 0, False, False),                         # whole tiles, everything visible
    ((129, 1, 1), (0, 40, 200), 8, 2, 64, 64, 33, 0, True, True),             # eight heads: one tile of the mix, partly empty
    ((17, 15, 100), (300, 0, 70), 5, 5, 24, 48, 40, 5, True, True),           # heads alone, key size below a step
    ((140,), (1000,), 32, 8, 64, 64, 100, 20, False, False),                  # a portion far behind the kept tokens
    ((150,), (90,), 32, 8, 64, 64, 128, 16, True, True),                      # kept tokens and a mix of 32 heads
    ((131,), (500,), 6, 2, 128, 32, 0, 0, False, False),                      # heads alone in waves of one workgroup and a half
    ((70, 66), (33, 2), 24, 6, 80, 112, 64, 3, True, True),                   # sizes between the instances
    ((160,), (0,), 8, 2, 128, 128, 1, 0, False, False),                       # a row sees itself alone
    ((130,), (0,), 32, 8, 128, 128, 50, 7, True, True),                       # the largest
    # keys split over workgroups: the sink in the first share, kept and window blocks in different ones, shares without a block
    ((150, 1), (700, 900), 32, 8, 64, 64, 512, 16, True, True),
    ((140,), (600,), 8, 2, 64, 64, 300, 20, True, True),
    ((135, 3), (800, 5), 32, 8, 64, 64, 400, 40, False, False),
    ((200, 1), (0, 2), 32, 8, 128, 128, 1024, 0, True, True),
    ((64,) + (1,) * 64, (10,) + tuple(range(300, 364)), 32, 8, 64, 64, 256, 0, False, False),
])
def test_tiles_are_the_attention(lens, starts, H, G, dk, dv, window, keep, sink, mixed):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(sum(lens) + H + dk)
    T, B, ps = sum(lens), len(lens), 8
    total = [s + n for s, n in zip(starts, lens)]
    pages = [-(-t // ps) for t in total]
    order = torch.randperm(sum(pages), generator=g)
    table = torch.full((B, max(pages) + 1), -1, dtype=torch.int32)
    for b in range(B):
        table[b, :pages[b]] = order[sum(pages[:b]):sum(pages[:b + 1])].int()
    kc = torch.randn(sum(pages), G, ps, dk, generator=g).bfloat16()
    vc = torch.randn(sum(pages), G, ps, dv, generator=g).bfloat16()
    q = (torch.randn(T + 2, H * dk + 8, generator=g) * 2).bfloat16()[:, :H * dk]
    mix = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g) if mixed else None
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    off = [sum(lens[:i]) for i in range(B)]
    item = i32([b for b, n in enumerate(lens) for _ in range(n)] + [-1, -1])
    pos = i32([s + i for s, n in zip(starts, lens) for i in range(n)] + [-1, 0])
    items = (item, i32(list(lens) + [0]), i32(off + [0]), i32(list(range(B)) + [-1]))
    scale = dk ** -0.5
    span = window + keep if window else 8 * table.shape[1]
    assert (K.sink_tile_splits(T + 2, B + 1, H, G, dk, dv, mixed, span) > 1) == (span >= 256)
    assert T >= 128 and K._lib().st_sink_tiles_fit(H, G, dk, dv, int(mixed), window, keep, table.shape[1], ps)
    args = (q.to(DEV), kc.to(DEV), vc.to(DEV), item, pos, table.to(DEV), H, scale)
    kw = dict(window=window, sink=sink, head_mix=mix.to(DEV) if mixed else None, keep_first=keep)
    got = K.sink_attention(*args, items=items, **kw).cpu().to(F64)
    rows = K.sink_attention(*args, **kw).cpu().to(F64)                        # the row kernel
    assert float(got[T:].abs().max()) == 0.0
    for b in range(B):
        idx = table[b, :pages[b]].long()
        flat = lambda c, w: c[idx].transpose(0, 1).reshape(G, -1, w)[:, :total[b]].to(F64).repeat_interleave(H // G, 0)
        k, v = flat(kc, dk), flat(vc, dv)
        r = slice(off[b], off[b] + lens[b])
        s = torch.einsum("ihd,hjd->hij", q[r].to(F64).reshape(-1, H, dk), k) * scale
        if mixed:
            s = torch.einsum("hg,gij->hij", mix.to(F64), s)
        i, j = torch.arange(starts[b], total[b])[:, None], torch.arange(total[b])[None]
        seen = (j <= i) & ((i - j < window) | (j < keep)) if window else j <= i
        s = s.masked_fill(~seen[None], float("-inf"))
        top = s.amax(-1, keepdim=True).clamp(min=0.0) if sink else s.amax(-1, keepdim=True)
        p = torch.exp(s - top)
        p = p / (p.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0))
        want = torch.einsum("hij,hjv->ihv", p, v).reshape(lens[b], -1)
        size = torch.einsum("hij,hjv->ihv", p, v.abs()).reshape(lens[b], -1)
        # the result is rounded to bfloat16 (2^-8 of it); a weight is off by its score's rounding (sums of up to 128 + 32 products
        # of numbers up to 40: 40 * 160 * 2^-24 = 4e-4 at most) and by 2^-17
        bound = 2.0 ** -8 * want.abs() + (4e-4 + 2.0 ** -17) * size + 1e-6
        assert bool(((got[r] - want).abs() <= bound).all()), float(((got[r] - want).abs() / bound).max())
        # and on the whole no further from it than the row kernel, whose weights are floats throughout
        err = lambda x: float((x[r] - want).norm() / want.norm())
        assert err(got) <= 1.05 * err(rows) + 1e-5, (err(got), err(rows))


def _attend(q, kc, vc, start, H, window, keep, sink, mix, tiles=True, scale=1.0):
    """One request whose T rows start at position ``start``; caches by whole pages in order."""
    from swifttransformer_amd.ops import kernels as K
    T = q.shape[0]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    item, pos = i32([0] * T), i32(list(range(start, start + T)))
    table = torch.arange(kc.shape[0], dtype=torch.int32, device=DEV)[None].contiguous()
    return K.sink_attention(q.to(DEV), kc.to(DEV), vc.to(DEV), item, pos, table, H, scale, window=window, sink=sink, keep_first=keep,
                            head_mix=mix.to(DEV) if mix is not None else None,
                            items=(item, i32([T]), i32([0]), i32([0])) if tiles else None)


@pytest.mark.parametrize("mixed", [False, True])
def test_scores_as_far_apart_as_floats_go(mixed):
    """Products of +-1.3e38: the weight of the smaller ones is e^-2.6e38, zero, whichever of the two a row (or a block of 32 keys)
    meets first."""
    H, d, ps, T = 4, 16, 16, 144
    g = torch.Generator().manual_seed(1)
    q, kc, vc = torch.zeros(T, H * d), torch.zeros(T // ps, H, ps, d), torch.randn(T // ps, H, ps, d, generator=g).bfloat16()
    q[:, ::d] = 1e19
    high = torch.rand(T, generator=g) < 0.3
    high[:40], high[40:72] = False, True                       # whole blocks of either kind
    kc[..., 0] = torch.where(high, 1.3e19, -1.3e19).view(T // ps, 1, ps)
    got = _attend(q.bfloat16(), kc.bfloat16(), vc, 0, H, 0, 0, False, torch.eye(H) if mixed else None).cpu().to(F64).view(T, H, d)
    v = vc.transpose(1, 2).reshape(T, H, d).to(F64)
    for i in range(T):
        best = high[:i + 1] if bool(high[:i + 1].any()) else ~high[:i + 1]
        want = v[:i + 1][best].mean(0)
        assert bool(((got[i] - want).abs() <= 2.0 ** -8 * want.abs() + 144 * 2.0 ** -22).all()), i


@pytest.mark.parametrize("H,G,dv,mixed,keep", [(32, 8, 64, False, 0), (5, 5, 48, False, 3), (8, 2, 128, True, 0), (32, 8, 64, True, 7)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_value_that_is_not_finite_reaches_the_rows_that_see_it_and_no_others(H, G, dv, mixed, keep, bad):
    """An infinity or NaN in one channel of one key head's value at position 75, in a key at position 90: rows before, rows behind the
    window and other channels are what they are without it; the rows and channels that see it are not finite."""
    dk, ps, T, window = 32, 16, 160, 50
    g = torch.Generator().manual_seed(H + dv)
    q = torch.randn(T, H * dk, generator=g).bfloat16()
    kc, vc = (torch.randn(T // ps, G, ps, w, generator=g).bfloat16() for w in (dk, dv))
    mix = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g) if mixed else None
    clean = _attend(q, kc, vc, 0, H, window, keep, True, mix, scale=dk ** -0.5).float().cpu().view(T, H, dv)
    v2 = vc.clone()
    v2[75 // ps, G - 1, 75 % ps, 7] = bad
    got = _attend(q, kc, v2, 0, H, window, keep, True, mix, scale=dk ** -0.5).float().cpu().view(T, H, dv)
    hit = torch.zeros(T, H, dv, dtype=torch.bool)
    hit[75:75 + window, H - H // G:, 7] = True
    assert not bool(got[hit].isfinite().any())
    # the same weights and values, summed in another order where a tile was made again (see the bound above)
    assert bool(((got - clean).abs() <= 2.0 ** -7 * clean.abs() + 4e-3)[~hit].all())
    k2 = kc.clone()
    k2[90 // ps, 0, 90 % ps, 3] = float("nan")
    got = _attend(q, k2, vc, 0, H, window, keep, True, mix, scale=dk ** -0.5).float().cpu().view(T, H, dv)
    hit = torch.zeros(T, H, dv, dtype=torch.bool)
    hit[90:90 + window, :H if mixed else H // G] = True
    assert not bool(got[hit].isfinite().any())
    assert bool(((got - clean).abs() <= 2.0 ** -7 * clean.abs() + 4e-3)[~hit].all())


@pytest.mark.parametrize("T,start,H,G,dk,dv,window,keep,sink,mixed,spread", [
    (512, 600, 32, 8, 64, 64, 1024, 0, True, True, 1), (512, 600, 32, 8, 64, 64, 1024, 16, False, False, 1),
    (700, 10, 32, 8, 128, 128, 300, 16, True, True, 1), (200, 900, 12, 3, 64, 64, 256, 0, True, True, 2),
    (300, 0, 8, 8, 80, 48, 0, 0, False, False, 3)])
def test_sums_before_the_rounding_are_no_further_from_float64_than_the_row_kernels(monkeypatch, T, start, H, G, dk, dv, window, keep, sink,
                                                                                   mixed, spread):
    """The float partial results of split keys, added up in float64: weights that met the values in fewer than 24 bits would show."""
    from swifttransformer_amd.ops import kernels as K
    made, make = [], K.empty
    monkeypatch.setattr(K, "empty", lambda *a: made.append(make(*a)) or made[-1])
    g = torch.Generator().manual_seed(T + H)
    ps, total = 16, start + T
    kc, vc = (torch.randn(-(-total // ps), G, ps, w, generator=g).bfloat16() for w in (dk, dv))
    q = (spread * torch.randn(T, H * dk, generator=g)).bfloat16()
    mix = torch.eye(H) + 0.1 * torch.randn(H, H, generator=g) if mixed else None

    def sums():
        o, ml = (t.to(F64) for t in made if t.dtype == torch.float32)
        o, m, l = o.view(T, -1, H, dv), ml[..., 0, None], ml[..., 1, None]
        w = torch.exp(m - m.amax(1, keepdim=True))
        return (w * torch.where(w > 0, o, 0.0)).sum(1) / (w * l).sum(1), o.shape[1]

    _attend(q, kc, vc, start, H, window, keep, sink, mix, scale=dk ** -0.5)
    tiles, splits = sums()
    assert splits > 1
    made.clear()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    item, pos = i32([0] * T), i32(list(range(start, total)))
    table = torch.arange(kc.shape[0], dtype=torch.int32, device=DEV)[None].contiguous()
    K.sink_attention(q.to(DEV), kc.to(DEV), vc.to(DEV), item, pos, table, H, dk ** -0.5, window=window, sink=sink, keep_first=keep,
                     head_mix=mix.to(DEV) if mixed else None, num_splits=splits)
    rows, _ = sums()
    flat = lambda c, w: c.to(DEV).transpose(0, 1).reshape(G, -1, w)[:, :total].to(F64).repeat_interleave(H // G, 0)
    k, v = flat(kc, dk), flat(vc, dv)
    s = torch.matmul(q.to(DEV).to(F64).view(T, H, dk).transpose(0, 1).contiguous(), k.transpose(1, 2).contiguous()) * dk ** -0.5
    if mixed:
        s = torch.matmul(mix.to(DEV).to(F64), s.reshape(H, -1)).view(s.shape)
    i, j = torch.arange(start, total, device=DEV)[:, None], torch.arange(total, device=DEV)[None]
    s = s.masked_fill(~((j <= i) & ((i - j < window) | (j < keep)) if window else j <= i), float("-inf"))
    top = s.amax(-1, keepdim=True).clamp(min=0.0) if sink else s.amax(-1, keepdim=True)
    p = torch.exp(s - top)
    want = torch.matmul(p / (p.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0)), v).transpose(0, 1)
    err = lambda x: float((x - want).norm() / want.norm())
    # (by a tenth to a half nearer; two bfloat16 numbers a weight: 1.4 to 7 times as far)
    assert err(tiles) <= err(rows), (err(tiles), err(rows))


def test_the_arena_has_room_for_the_shares_of_smaller_steps():
    """Steps of fewer rows split their keys more ways: their partial results fit what was measured on the largest step, which splits none."""
    from swifttransformer_amd.ops import arena
    from swifttransformer_amd.ops import kernels as K
    H, G, d, ps, most = 8, 2, 64, 16, 6144
    kc = torch.randn(1, G, ps, d, device=DEV).bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table = torch.zeros(1, 64, dtype=torch.int32, device=DEV)
    a = arena.StepArena(DEV)

    def run(T):
        item, pos = torch.zeros(T, dtype=torch.int32, device=DEV), torch.arange(T, dtype=torch.int32, device=DEV) % 1024
        q = torch.zeros(T, H * d, dtype=torch.bfloat16, device=DEV)
        with arena.using(a):
            K.sink_attention(q, kc, kc, item, pos, table, H, 1.0, window=1024, items=(item, i32([min(T, 1024)]), i32([0]), i32([0])))
        torch.cuda.synchronize()

    assert K.sink_tile_splits(most, 1, H, G, d, d, False, 1024) == 1
    a.measure = True
    run(most)
    a.measure = False
    a.resize(a.peak)
    for T in (128, 512, 1000, 2048, 2500, 3000, 4000, most):
        run(T)
    assert a.overflows == 0
