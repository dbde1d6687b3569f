"""The experts' choices, weights and sorted lists against a plain walk in float64: every rule, outputs up to and past 16, 32 and 64, rows
around what one workgroup routes, ties, identity experts, padding rows, logits of equal size and infinities."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _plain(z, correction, scale, top, mode, groups, keep):
    """One token's choices and weights; ties go to the lower index."""
    E = len(z)
    sig = torch.sigmoid(z)
    soft = torch.softmax(z, 0)
    by = {0: z, 1: z, 2: z, 3: sig + correction, 4: soft + correction}[mode].tolist()
    allowed = list(range(E))
    if mode == 2 and keep < groups:
        per = E // groups
        best = sorted(range(groups), key=lambda g: (-max(by[g * per:(g + 1) * per]), g))[:keep]
        allowed = [e for e in allowed if e // per in best]
    ids = sorted(allowed, key=lambda e: (-by[e], e))[:top]
    if mode == 0:
        w = sig[ids]
    elif mode == 1:
        w = torch.softmax(z[ids], 0)
    elif mode == 3:
        w = sig[ids] / (sig[ids].sum() + 1e-20) * scale
    else:
        w = soft[ids]
    return ids, w


@pytest.mark.parametrize("T,E,identity,top,mode,groups,keep", [
    (1, 16, 0, 2, 3, 1, 1), (64, 16, 0, 16, 0, 1, 1), (65, 16, 0, 2, 2, 4, 2), (7, 1, 0, 1, 1, 1, 1), (32, 17, 0, 5, 1, 1, 1),
    (33, 32, 0, 3, 2, 8, 8), (16, 64, 0, 8, 2, 8, 3), (17, 60, 4, 6, 4, 1, 1), (24, 14, 2, 2, 4, 1, 1), (300, 12, 0, 4, 2, 3, 2),
    (5, 65, 0, 2, 3, 1, 1), (130, 100, 3, 4, 4, 1, 1)])
def test_routes_and_lists(T, E, identity, top, mode, groups, keep):
    from swifttransformer_amd.ops import kernels as K
    lib, ptr = K._lib(), K._ptr
    g = torch.Generator().manual_seed(T * 7 + E)
    out = E + identity
    z = torch.randn(T, out + 3, generator=g)
    z[0, :out] = 0.5                                           # all the same: the lowest indices
    if T > 4 and out > 1:
        z[2, out // 2] = float("-inf")
    correction = torch.randn(out, generator=g) * 0.2
    if mode >= 3:
        correction[:] = correction.round(decimals=2)
        z[0, :out] += 0.01 * torch.arange(out)                 # (shares of equal logits differ by the order of a sum alone)
    item = torch.zeros(T, dtype=torch.int32)
    if T > 4:
        item[T - 2] = -1
    dev = lambda t: t.to("cuda")
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device="cuda")
    tile = 16
    cap = K.moe_capacity(T, top, E, tile)
    ids, srt, place, texp = i32(T * top), i32(cap), i32(T * top), i32(cap // tile)
    w = torch.full((T * top,), -7.0, device="cuda")
    zd, cd, it = dev(z), dev(correction), dev(item)
    if K.moe_routes_at_once(T, out):
        K._check(lib.st_moe_route_align(ptr(ids), ptr(w), ptr(srt), ptr(place), ptr(texp), ptr(zd), out + 3, ptr(it), ptr(cd), 1.5, T, out, E,
                                        top, mode, groups, keep, cap, tile, K._stream()))
    else:
        K._check(lib.st_moe_route(ptr(ids), ptr(w), ptr(zd), out + 3, ptr(it), ptr(cd), 1.5, T, out, top, mode, groups, keep, K._stream()))
        K._check(lib.st_moe_align(ptr(srt), ptr(place), ptr(texp), ptr(ids), T * top, E, cap, tile, K._stream()))
    ids, w, srt, place, texp = (t.cpu() for t in (ids.view(T, top), w.view(T, top), srt, place.view(T, top), texp))
    for t in range(T):
        if item[t] < 0:
            assert (ids[t] == -1).all() and (w[t] == 0).all() and (place[t] == -1).all()
            continue
        want, ww = _plain(z[t, :out].double(), correction.double(), 1.5, top, mode, groups, keep)
        assert ids[t].tolist() == want, (t, ids[t], want)
        # a handful of float operations on numbers up to one (times 1.5)
        assert float((w[t].double() - ww).abs().max()) <= 16 * 2.0 ** -24
    # every pair of an expert with weights has a place of its own in a tile of that expert, every other place is empty
    real = (ids >= 0) & (ids < E)
    assert (place[~real] == -1).all()
    p = place[real].long()
    assert p.unique().numel() == p.numel() == int((srt >= 0).sum())
    assert torch.equal(srt[p], torch.arange(T * top, dtype=torch.int32).view(T, top)[real])
    assert torch.equal(texp[p // tile], ids[real])
    used = int((texp >= 0).sum())
    assert (texp[:used] >= 0).all() and (texp[1:used] >= texp[:used - 1]).all()        # an expert's tiles are neighbours


def test_no_token_leaves_no_tile():
    """Routing and sorting of no token marks every place and tile as empty, as sorting alone does: the products that follow read them."""
    from swifttransformer_amd.ops import kernels as K
    E, tile, lib, P = 8, 16, K._lib(), K._ptr
    cap = K.moe_capacity(0, 2, E, tile)
    i32 = lambda n: torch.full((n,), 5, dtype=torch.int32, device="cuda")
    order, place, owner, ids = i32(cap), i32(2), i32(cap // tile), i32(2)
    wts, logits = torch.ones(2, device="cuda"), torch.zeros(1, E, device="cuda")
    K._check(lib.st_moe_route_align(P(ids), P(wts), P(order), P(place), P(owner), P(logits), E, None, None, 1.0, 0, E, E, 2, 1, 1, 1, cap, tile,
                                    K._stream()))
    assert bool((order == -1).all()) and bool((owner == -1).all())
