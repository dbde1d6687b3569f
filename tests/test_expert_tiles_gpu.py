"""Routed experts in tiles of 64 and 128 places (bfloat16): row counts around a tile, feature counts and depths that leave part of a
block or of a step, experts without a pair, one expert with all of them, padding rows, every unit and the single-choice sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu
F64 = torch.float64


def _experts(x, ids, weights, wg, wu, wd, unit, on_input, limit):
    """float64 sums of a token's experts, and of their absolute values (what the rounding is relative to)."""
    out, size = torch.zeros(x.shape[0], wd.shape[1], dtype=F64), torch.zeros(x.shape[0], wd.shape[1], dtype=F64)
    for j in range(ids.shape[1]):
        for e in ids[:, j].unique().tolist():
            rows = (ids[:, j] == e).nonzero()[:, 0]
            s = weights[rows, j][:, None]
            h = x[rows] * s if on_input else x[rows]
            u = h @ wu[e].T
            if unit == "gelu":
                y = 0.5 * u * (1 + torch.erf(u / 2 ** 0.5))
            else:
                g = h @ wg[e].T
                if unit == "silu":
                    y = g * torch.sigmoid(g) * u
                else:
                    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
                    y = g * torch.sigmoid(1.702 * g) * (u + 1)
            y = y if on_input else y * s
            out[rows] += y @ wd[e].T
            size[rows] += y.abs() @ wd[e].abs().T
    return out, size


@pytest.mark.parametrize("T,W,F,E,top,style,clamped,same", [
    (64, 64, 64, 3, 2, "softmax_output", False, False),
    (65, 136, 72, 5, 2, "scaled_input", False, False),        # depths of 136 and 72: two whole steps and one, and 8 more
    (127, 8, 200, 4, 1, "scaled_input", False, True),         # a depth below one step; one choice a token: straight into the stream
    (128, 200, 8, 2, 2, "softmax_output", False, False),
    (129, 72, 130 * 8, 3, 1, "sigmoid_output", False, True),  # one expert has 129 rows, the others none
    (500, 264, 328, 4, 3, "softmax_corrected", True, False),
    (333, 96, 160, 9, 2, "sigmoid_output", False, False),
    (1100, 128, 96, 300, 8, "softmax_output", False, False),  # more tiles than a wave has lanes
])
def test_tiles_of_64_and_128_places(T, W, F, E, top, style, clamped, same):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(T + W + F)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).bfloat16().to(F64)
    x, wu, wd = rnd(T, W), rnd(E, F, W, std=W ** -0.5), rnd(E, W, F, std=F ** -0.5)
    gated = style != "sigmoid_output"
    wg = rnd(E, F, W, std=W ** -0.5) if gated else None
    z = torch.randn(T, E, generator=g) * 2
    if same:
        z = torch.arange(E, dtype=torch.float32).flip(0).repeat(T, 1)
    limit = 0.9
    corrected = style in ("sigmoid_output", "softmax_corrected")
    correction = torch.randn(E, generator=g) if corrected else None
    zd = z.to(F64)
    score = {"scaled_input": torch.sigmoid(zd), "softmax_output": zd, "sigmoid_output": torch.sigmoid(zd),
             "softmax_corrected": torch.softmax(zd, 1)}[style]
    ids = torch.topk(score + (correction.to(F64) if corrected else 0), top, dim=1).indices
    wts = score.gather(1, ids)
    if style == "softmax_output":
        wts = torch.softmax(wts, 1)
    elif style == "sigmoid_output":
        wts = wts / wts.sum(1, keepdim=True) * 1.5
    unit = "gelu" if not gated else "clamped" if clamped or style == "scaled_input" else "silu"
    want, size = _experts(x, ids, wts, wg, wu, wd, unit, style == "scaled_input", limit)
    dev = lambda t, d=torch.bfloat16: None if t is None else t.to("cuda").to(d)
    res = torch.randn(T, W, generator=g)
    item = torch.zeros(T, dtype=torch.int32, device="cuda")
    item[T - 3:] = -1                                          # padding rows keep what they held
    r = dev(res, torch.float32)
    got = K.routed_experts(dev(x), dev(z, torch.float32), dev(wg), dev(wu), dev(wd), r, top=top, limit=limit, out_scale=0.5,
                           token_item=item, style=style, clamped=clamped, correction=dev(correction, torch.float32), scale=1.5)
    assert K.moe_tile(T, top, E, True) in (64, 128)
    # an expert's inner values are rounded to bfloat16 once (8 significant bits: by 2^-8 of each at most); every sum is float
    bound = 0.5 * (2.0 ** -8 + 1e-4) * size + 1e-5
    err = (got.double().cpu() - (res.to(F64) + 0.5 * want)).abs()
    assert bool((err[:T - 3] <= bound[:T - 3]).all()), float((err / bound)[:T - 3].max())
    assert torch.equal(got[T - 3:].cpu(), res[T - 3:])


@pytest.mark.parametrize("E,W,F,T,top", [(16, 256, 264, 100, 2), (16, 256, 1000, 60, 2), (8, 128, 2048, 64, 2), (4, 128, 8192, 30, 1), (8, 128, 768, 120, 4)])
def test_sums_of_64_places_are_no_further_from_float64_than_those_of_16(E, W, F, T, top):
    """The output products of the same rows in tiles of 64 places and of 16, whose waves share the depth in short chains."""
    from swifttransformer_amd.ops import kernels as K
    dev, P, lib = "cuda", K._ptr, K._lib()
    g = torch.Generator(device=dev).manual_seed(F)
    ids = torch.stack([torch.randperm(E, generator=g, device=dev)[:top] for _ in range(T)]).int().reshape(-1)
    w = (torch.randn(E, W, F, generator=g, device=dev) * 0.02).bfloat16()
    rows = torch.randn(T * top, F, generator=g, device=dev).bfloat16()
    want = torch.stack([w[e].to(torch.float64) @ rows[i].to(torch.float64) for i, e in enumerate(ids.tolist())])

    def err(tile):
        cap = K.moe_capacity(T, top, E, tile)
        i32 = lambda n: torch.empty(n, dtype=torch.int32, device=dev)
        order, place, owner = i32(cap), i32(T * top), i32(cap // tile)
        K._check(lib.st_moe_align(P(order), P(place), P(owner), P(ids), T * top, E, cap, tile, K._stream()))
        y = torch.zeros(cap, F, dtype=torch.bfloat16, device=dev)
        y[place.long()] = rows
        out = torch.empty(cap, W, device=dev)
        K._check(lib.st_moe_down(None, None, P(out), P(y), P(w), P(order), P(owner), cap, tile, 2, W, F, 1.0, K.dtype_code(y.dtype), K._stream()))
        return float((out[place.long()] - want).norm() / want.norm())

    assert err(64) <= err(16), (err(64), err(16))


@pytest.mark.parametrize("W,F", [(64, 128), (128, 136), (192, 256), (200, 264), (320, 520)])      # depths of 1 to 5 steps, 4 of them part of a step
@pytest.mark.parametrize("counts", [(1, 127, 0, 260), (32, 33, 64, 300), (65, 96, 97, 200), (128, 129, 160, 31)])
def test_last_tiles_that_are_partly_empty(W, F, counts):
    """Experts with chosen numbers of rows (one choice a token), around every block of 32 places of their last tile of 128."""
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(W + sum(counts))
    E, T = len(counts), sum(counts)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).bfloat16().to(F64)
    x, wg, wu, wd = rnd(T, W), rnd(E, F, W, std=W ** -0.5), rnd(E, F, W, std=W ** -0.5), rnd(E, W, F, std=F ** -0.5)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)]
    z = torch.full((T, E), -4.0)
    z[torch.arange(T), ids] = 4.0
    dev = lambda t, d=torch.bfloat16: t.to("cuda").to(d)
    res = torch.randn(T, W, generator=g)
    for top in (1, 2):                                         # straight into the stream; a row a pair (the second choice: expert 0 or 1)
        ids2 = torch.topk(z, top, dim=1).indices
        wts = torch.softmax(z.to(F64).gather(1, ids2), 1)
        want, size = _experts(x, ids2, wts, wg, wu, wd, "silu", False, 0.0)
        got = K.routed_experts(dev(x), dev(z, torch.float32), dev(wg), dev(wu), dev(wd), dev(res, torch.float32), top=top, style="softmax_output")
        assert K.moe_tile(T, top, E, True) == (128 if top * T >= 112 * E else 64)
        # an expert's inner values are rounded to bfloat16 once (by 2^-8 of each at most); every sum is float
        err = (got.double().cpu() - (res.to(F64) + want)).abs()
        assert bool((err <= (2.0 ** -8 + 1e-4) * size + 1e-5).all()), float((err / size).max())


@pytest.mark.parametrize("W,F,up,down", [
    (840, 440, "one", "one"), (1160, 648, "wide", "wide"), (64, 712, "wide", "two"), (1224, 64, "two", "wide"), (128, 392, "one", "two"),
    (776, 136, "two", "one"), (1096, 712, "wide", "wide")])
@pytest.mark.parametrize("unit", ["silu", "gelu"])
def test_tiles_of_128_places_on_as_many_weight_rows_as_fill_the_chip(W, F, up, down, unit):
    """24 experts with chosen numbers of rows: 256 weight rows a workgroup ("wide"), or 128 with one or two steps of loads ahead; depths of 1
    to 20 steps, whole and not, feature counts that leave part of a block."""
    from swifttransformer_amd.ops import kernels as K
    counts = (1, 127, 0, 260, 32, 33, 64, 300, 65, 96, 97, 200, 128, 129, 160, 31, 256, 255, 2, 180, 140, 111, 63, 190)
    g = torch.Generator().manual_seed(W + F)
    E, T = len(counts), sum(counts)
    cap = K.moe_capacity(T, 1, E, 128)
    assert K.moe_tile(T, 1, E, True) == 128
    units = torch.cuda.get_device_properties(0).multi_processor_count
    form = lambda blocks: "two" if cap // 128 * blocks <= units else "one" if 7 * (cap // 128) * blocks <= 10 * units else "wide"
    if unit == "silu":
        assert (form(-(-F // 64)), form(-(-W // 128))) == (up, down)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).bfloat16().to(F64)
    x, wu, wd = rnd(T, W), rnd(E, F, W, std=W ** -0.5), rnd(E, W, F, std=F ** -0.5)
    wg = rnd(E, F, W, std=W ** -0.5) if unit == "silu" else None
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)]
    z = torch.full((T, E), -4.0)
    z[torch.arange(T), ids] = 4.0
    dev = lambda t, d=torch.bfloat16: None if t is None else t.to("cuda").to(d)
    res = torch.randn(T, W, generator=g)
    want, size = _experts(x, ids[:, None], torch.ones(T, 1, dtype=F64), wg, wu, wd, unit, False, 0.0)
    got = K.routed_experts(dev(x), dev(z, torch.float32), dev(wg), dev(wu), dev(wd), dev(res, torch.float32), top=1, style="softmax_output")
    # an expert's inner values are rounded to bfloat16 once (by 2^-8 of each at most); every sum is float
    err = (got.double().cpu() - (res.to(F64) + want)).abs()
    assert bool((err <= (2.0 ** -8 + 1e-4) * size + 1e-5).all()), float((err / size).max())
