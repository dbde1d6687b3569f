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


@pytest.mark.parametrize("T,W,E,identity,top,mode,groups,keep,biased", [
    (1, 768, 16, 0, 2, 3, 1, 1, False), (16, 8, 5, 0, 2, 1, 1, 1, True), (17, 1024, 16, 0, 2, 2, 4, 2, False), (32, 1000, 14, 2, 2, 4, 1, 1, False),
    (16, 1096, 32, 0, 3, 0, 1, 1, True), (3, 40, 17, 0, 4, 1, 1, 1, False), (8, 2048, 16, 0, 2, 2, 4, 2, False)])
def test_the_routers_product_and_its_routes_in_one_kernel(T, W, E, identity, top, mode, groups, keep, biased):
    """Whole numbers, whose products and sums are exact: the same choices, weights and places per expert as from the logits themselves."""
    from swifttransformer_amd.ops import kernels as K
    lib, ptr = K._lib(), K._ptr
    g = torch.Generator().manual_seed(T + W)
    out = E + identity
    rows = -(-out // 8) * 8
    x = torch.randint(-2, 3, (T, W), generator=g).float() * (torch.rand(T, W, generator=g) < 8 / W)        # (logits of some units)
    w = torch.randint(-3, 4, (rows, W), generator=g).float()
    bias = torch.randint(-2, 3, (rows,), generator=g).float() / 4 if biased else None
    z = x @ w.T + (bias if biased else 0)
    correction = torch.randn(out, generator=g) * 0.2
    item = torch.zeros(T, dtype=torch.int32)
    if T > 4:
        item[T - 2] = -1
    cap = K.moe_capacity(T, top, E, 16)
    dev = lambda t, d: t.to("cuda").to(d)
    xd, wd, zd, cd, it = dev(x, torch.bfloat16), dev(w, torch.bfloat16), dev(z, torch.float32), dev(correction, torch.float32), item.to("cuda")
    bd = dev(bias, torch.float32) if biased else None
    assert K.moe_routes_by_matrix(xd, wd, out)

    def run(by_matrix):
        i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device="cuda")
        ids, srt, place, texp, wts = i32(T * top), i32(cap), i32(T * top), i32(cap // 16), torch.full((T * top,), -7.0, device="cuda")
        tail = (T, out, E, top, mode, groups, keep, cap, 16, K._stream())
        if by_matrix:
            K._check(lib.st_moe_router_align(ptr(ids), ptr(wts), ptr(srt), ptr(place), ptr(texp), ptr(xd), ptr(wd), ptr(bd), W, rows, ptr(it), ptr(cd),
                                             1.5, *tail))
        else:
            K._check(lib.st_moe_route_align(ptr(ids), ptr(wts), ptr(srt), ptr(place), ptr(texp), ptr(zd), rows, ptr(it), ptr(cd), 1.5, *tail))
        return [t.cpu() for t in (ids, wts, texp, srt, place)]
    (ids, wts, texp, srt, place), (ids0, wts0, texp0, srt0, _p) = run(True), run(False)
    assert torch.equal(ids, ids0) and torch.equal(wts, wts0) and torch.equal(texp, texp0)
    assert torch.equal(srt.view(-1, 16).sort(1).values, srt0.view(-1, 16).sort(1).values)       # (places within a tile are in any order)
    real = (ids >= 0) & (ids < E)
    assert torch.equal(srt[place[real].long()], torch.arange(T * top, dtype=torch.int32)[real]) and bool((place[~real] == -1).all())


def test_larger_routers_keep_kernels_of_their_own():
    from swifttransformer_amd.ops import kernels as K
    offered = lambda T, W, out, dt=torch.bfloat16: K.moe_routes_by_matrix(torch.empty(T, W, dtype=dt, device="cuda"),
                                                                          torch.empty(-(-out // 8) * 8, W, dtype=dt, device="cuda"), out)
    assert offered(16, 2048, 16) and not offered(17, 2048, 16) and not offered(33, 64, 16) and not offered(17, 64, 17)
    assert not offered(1, 64, 33) and not offered(1, 60, 16) and not offered(1, 64, 16, torch.float32) and not offered(0, 64, 16)
