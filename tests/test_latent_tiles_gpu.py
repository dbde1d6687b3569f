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
    # weights are rounded to bfloat16 before they meet the entries and are summed as rounded (2^-9 each way), the result once (2^-9)
    err = (out.view(tokens, heads, entry).to(F64) - want).abs()
    assert bool((err <= 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-4).all()), float((err / size).max())


def test_wide_block_tables_do_not_fit():
    from swifttransformer_amd.ops import kernels as K
    assert K.latent_tiles_fit(32, 160, 16, 128, 16) and K.latent_tiles_fit(32, 256, 16, 2048, 16)
    assert not K.latent_tiles_fit(32, 160, 16, 40000, 16) and not K.latent_tiles_fit(32, 272, 16, 8)
