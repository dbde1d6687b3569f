"""Tiles over a latent cache as latent attention with large entries takes them: few workgroups, whose keys two groups of waves share, and many."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


@pytest.mark.parametrize("heads,entry,window", [(4, 144, 0), (32, 160, 0), (12, 160, 50), (3, 256, 0), (16, 192, 100)])
@pytest.mark.parametrize("start,tokens", [(0, 1), (0, 64), (37, 65), (500, 3), (130, 130), (0, 900)])
def test_tiles_of_latent_entries(heads, entry, window, start, tokens):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(entry + tokens)
    ps, n, scale = 16, start + tokens, 0.1
    pages = -(-n // ps)
    cache = torch.randn(pages + 1, 1, ps, entry, generator=g, device=DEV).bfloat16()
    cache[-1] = float("nan")                                   # nobody's page
    order = torch.randperm(pages, generator=g, device=DEV).int()
    q = torch.randn(tokens, heads * entry, generator=g, device=DEV).bfloat16()
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    q0 = list(range(0, tokens, 64)) + [0]
    item = i32(*([0] * (len(q0) - 1)), -1)                     # and a padding entry
    out = torch.empty(tokens, heads * entry, dtype=torch.bfloat16, device=DEV)
    sh = K.LatentShape(heads, entry, entry, scale, 0, None, 1.0, None, window)
    K.latent_tiles(q, cache, item, i32(*q0), i32(0), i32(start), i32(tokens), order.view(1, -1), sh, out)
    keys = cache[order.long()].reshape(-1, entry)[:n].to(F64)
    i, j = torch.arange(start, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    seen = (j <= i) & ((i - j < window) if window else torch.ones_like(j, dtype=torch.bool))
    s = torch.matmul(q.view(tokens, heads, entry).to(F64).transpose(0, 1), keys.T) * scale
    p = torch.softmax(s.masked_fill(~seen[None], float("-inf")), -1)
    want, size = torch.matmul(p, keys).transpose(0, 1), torch.matmul(p, keys.abs()).transpose(0, 1)
    # weights are rounded to bfloat16 before they meet the entries (by 2^-8 at most) and summed as rounded, which takes the mean of their
    # errors out again; the result is rounded once (2^-8)
    err = (out.view(tokens, heads, entry).to(F64) - want).abs()
    assert bool((err <= 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-4).all()), float((err / size).max())


@pytest.mark.parametrize("heads,entry,tokens", [(4, 160, 64), (32, 144, 1000), (6, 256, 40)])       # two groups of waves, one, two
def test_the_normaliser_is_the_sum_of_unrounded_weights(heads, entry, tokens):
    """A coordinate that only the first key's entry has, whose weight is exactly one: its result is one over the normaliser, and nothing
    but the result's own rounding separates it from float64."""
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(heads + entry)
    ps, start = 16, 70
    n = start + tokens
    pages = -(-n // ps)
    cache = torch.zeros(pages * ps, entry, device=DEV)
    cache[0, 0], cache[1:, 1] = 1.0, -1.0                      # scores: the first key's 0, all others' -a
    cache = cache.view(pages, 1, ps, entry).bfloat16()
    q = torch.zeros(tokens, heads, entry, device=DEV)
    q[..., 1] = 0.01 + torch.rand(tokens, heads, generator=g, device=DEV)
    q = q.view(tokens, -1).bfloat16()
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    q0 = list(range(0, tokens, 64))
    out = torch.empty(tokens, heads * entry, dtype=torch.bfloat16, device=DEV)
    bt = torch.arange(pages, device=DEV, dtype=torch.int32).view(1, -1)
    K.latent_tiles(q, cache, i32(*([0] * len(q0))), i32(*q0), i32(0), i32(start), i32(tokens), bt,
                   K.LatentShape(heads, entry, entry, 1.0, float_sum=True), out)
    a = q.view(tokens, heads, entry)[..., 1].to(F64)
    others = torch.arange(start, n, device=DEV, dtype=F64)[:, None]                # keys beside the first one
    want = 1.0 / (1.0 + others * torch.exp(-a))
    err = (out.view(tokens, heads, entry)[..., 0].to(F64) - want).abs() / want
    # the rounding of the result, up to 1,070 float additions and the hardware's exponentials; equal weights rounded to bfloat16 would all
    # be off to the same side, by up to 2^-8 more
    assert float(err.max()) <= 2.0 ** -8 + 1100 * 2.0 ** -24, float(err.max())


# a launch of few tiles shares out their keys over two groups of waves; with many (here: entries that are skipped), or with page lists that leave
# no room for two groups' blocks, one group goes through all of a tile's keys
@pytest.mark.parametrize("skipped,long_list", [(0, False), (400, False), (0, True)])
@pytest.mark.parametrize("entry,heads,rot_off,pairs,window,scale,float_sum", [
    (64, 5, 40, 9, 0, 0.2, False), (128, 3, 96, 16, 70, -0.1, False), (160, 4, 128, 16, 0, 0.1, True), (144, 6, 136, 4, 33, -0.15, True),
    (192, 2, 0, 5, 100, 0.1, True), (256, 3, 240, 8, 0, 0.08, True), (160, 4, 128, 16, 40, 0.1, False)])
def test_tiles_with_turned_pairs_sinks_and_windows(entry, heads, rot_off, pairs, window, scale, float_sum, skipped, long_list):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(entry + heads)
    ps, start, tokens = 16, 90, 150
    n, out_dim = start + tokens, entry - 16
    pages = -(-n // ps)
    listed = {64: 35000, 128: 30000, 256: 20000}.get(entry, 24000) if long_list else pages
    cache = torch.randn(pages + 1, 1, ps, entry, generator=g, device=DEV).bfloat16()
    cache[-1] = float("nan")                                   # nobody's page, listed behind the request's own
    order = torch.randperm(pages, generator=g, device=DEV).int()
    bt = torch.full((1, listed), pages, dtype=torch.int32, device=DEV)
    bt[0, :pages] = order
    q = torch.randn(tokens, heads, entry, generator=g, device=DEV).bfloat16()
    freq = torch.rand(pairs, generator=g, device=DEV)
    sink = torch.randn(heads, generator=g, device=DEV)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    q0 = [0] * skipped + list(range(0, tokens, 64))
    item = [-1] * skipped + [0] * (len(q0) - skipped)
    out = torch.empty(tokens, heads * out_dim, dtype=torch.bfloat16, device=DEV)
    K.latent_tiles(q.view(tokens, -1), cache, i32(*item), i32(*q0), i32(0), i32(start), i32(tokens), bt,
                   K.LatentShape(heads, entry, out_dim, scale, rot_off, freq, 1.25, sink, window, float_sum), out)
    keys = cache[order.long()].reshape(-1, entry)[:n].to(F64)
    i, j = torch.arange(start, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    seen = (j <= i) & ((i - j < window) if window else torch.ones_like(j, dtype=torch.bool))
    angle = (torch.arange(start, n, device=DEV).float()[:, None] * freq[None]).to(F64)[:, None]          # (float angles)
    c, s = torch.cos(angle) * 1.25, torch.sin(angle) * 1.25
    turned = q.to(F64)
    even, odd = turned[..., rot_off:rot_off + 2 * pairs:2].clone(), turned[..., rot_off + 1:rot_off + 2 * pairs:2].clone()
    turned[..., rot_off:rot_off + 2 * pairs:2], turned[..., rot_off + 1:rot_off + 2 * pairs:2] = even * c - odd * s, odd * c + even * s
    turned = turned.bfloat16().to(F64)
    z = torch.matmul(turned.transpose(0, 1), keys.T) * scale
    z = torch.cat([z.masked_fill(~seen[None], float("-inf")), sink.to(F64)[:, None, None].expand(heads, tokens, 1)], 2)
    p = torch.softmax(z, -1)[..., :-1]
    want, size = torch.matmul(p, keys[:, :out_dim]).transpose(0, 1), torch.matmul(p, keys[:, :out_dim].abs()).transpose(0, 1)
    # a weight is rounded to bfloat16 (2^-8 at most) and so is the result; a turned number may be rounded to the other side than here (2^-8 of
    # up to 6, against a key of up to 5, times the scale: a score off by 0.12 |scale|)
    err = (out.view(tokens, heads, out_dim).to(F64) - want).abs()
    assert bool((err <= (2.0 ** -8 + 0.24 * abs(scale)) * size + 2.0 ** -8 * want.abs() + 1e-4).all()), float((err / size).max())


def test_float_normalisers_are_offered_for_large_entries_alone():
    from swifttransformer_amd.ops import kernels as K
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    cache, q = torch.zeros(1, 1, 16, 128, device=DEV).bfloat16(), torch.zeros(4, 128, device=DEV).bfloat16()
    with pytest.raises(K.KernelError, match="float normalisers"):
        K.latent_tiles(q, cache, i32(0), i32(0), i32(0), i32(0), i32(4), i32(0).view(1, 1), K.LatentShape(1, 128, 128, 1.0, float_sum=True),
                       torch.empty_like(q))


def test_wide_block_tables_do_not_fit():
    from swifttransformer_amd.ops import kernels as K
    assert K.latent_tiles_fit(32, 160, 16, 128, 16) and K.latent_tiles_fit(32, 256, 16, 2048, 16)
    assert not K.latent_tiles_fit(32, 160, 16, 40000, 16) and not K.latent_tiles_fit(32, 272, 16, 8)
