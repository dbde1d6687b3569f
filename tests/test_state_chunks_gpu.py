"""The additive recurrence by chunks, and by the walk of short items, against the recurrence in float64: items of 1 row to several chunks
around the limits of a walk (16) and of a chunk (64), heads that share queries and keys, sizes with and without whole 16-byte pieces,
states that are parts of larger ones, decays of exactly 0 and 1, one row of gates for all tokens, and a portion that goes on from the
state another one left."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64
# the roundings on a number's way: up to 128 + 64 products and sums, 64 decays of the walk or a few of the chunks, in units of 2^-24
# of the sum of magnitudes
UNIT = 512 * 2.0 ** -24
i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)


def _walk(q, k, v, a, b, skip, S):
    out = torch.empty(v.shape, dtype=F64)
    for t in range(q.shape[0]):
        S = b[t][:, None, None] * S + (a[t][:, None] * k[t])[:, :, None] * v[t][:, None, :]
        out[t] = (S * q[t][:, :, None]).sum(1) + skip[:, None] * v[t]
    return out, S


@pytest.mark.parametrize("lens,heads,groups,kd,vd,gates", [
    ((1, 15, 16, 17, 63), 4, 2, 64, 64, "rows"), ((64, 65, 1, 129), 2, 1, 64, 128, "rows"), ((200, 2), 3, 3, 5, 7, "rows"),
    ((33, 80, 3), 6, 3, 80, 48, "rows"), ((130, 16), 2, 1, 128, 128, "rows"), ((17, 16, 3), 2, 2, 128, 100, "rows"),
    ((1,) * 70, 2, 2, 64, 32, "rows"), ((70,) + (1,) * 66, 2, 1, 16, 16, "rows"), ((1, 1, 1), 2, 1, 128, 128, "rows"),
    ((1,) * 5, 4, 4, 64, 128, "one"), ((1,) * 3, 2, 2, 20, 100, "one"), ((90, 7), 4, 4, 64, 64, "one")])
def test_chunks_are_the_recurrence(lens, heads, groups, kd, vd, gates):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(sum(lens) + kd)
    T, B = sum(lens) + 2, len(lens) + 1                        # two rows of no item; one padding item
    x = torch.randn(T, 2 * groups * kd + heads * vd + (3 if kd == 5 else 0), generator=g)
    rows = 1 if gates == "one" else T
    step = torch.rand(rows, heads, generator=g) * 0.1 + 0.001
    decay = torch.exp(-16 * torch.rand(rows, heads, generator=g) * step)
    if rows > 1:
        decay[::7, 0] = 1.0
        decay[min(40, T - 3), -1] = 0.0
        decay[0, 0] = 0.0
    else:
        decay[0, 0] = 1.0
    skip = torch.randn(heads, generator=g) if kd != 20 else None
    whole = torch.randn(B + 2, heads * kd * vd + 12, generator=g)
    off = [sum(lens[:i]) for i in range(len(lens))]
    slots = list(range(len(lens), 0, -1))                      # slot 0 and the last stay untouched
    items = (None, i32(list(lens) + [0]), i32(off + [0]), i32(slots + [-1]))
    d, st = x.to(DEV), whole.to(DEV)
    cut = [0, groups * kd, 2 * groups * kd, 2 * groups * kd + heads * vd]
    q, k, v = (d[:, lo:hi] for lo, hi in zip(cut, cut[1:]))
    y = K.state_scan(q, k, v, step.to(DEV), decay.to(DEV), st[:, 12:].unflatten(1, (heads, kd, vd)), items, heads, "additive",
                     skip=skip.to(DEV) if skip is not None else None, max_item_rows=1 if max(lens) == 1 else 0, chunks=True)
    f = lambda t, n, w: t.cpu().to(F64).reshape(T, n, w).repeat_interleave(heads // n, 1)
    q6, k6, v6 = f(q, groups, kd), f(k, groups, kd), f(v, heads, vd)
    a6, b6 = step.to(F64).expand(T, heads), decay.to(F64).expand(T, heads)
    s6 = skip.to(F64) if skip is not None else torch.zeros(heads, dtype=F64)
    was = whole[:, 12:].reshape(-1, heads, kd, vd).to(F64)
    now = st[:, 12:].cpu().to(F64).reshape(was.shape)
    for n, lo, slot in zip(lens, off, slots):
        r = slice(lo, lo + n)
        o, S = _walk(q6[r], k6[r], v6[r], a6[r], b6[r], s6, was[slot])
        oa, Sa = _walk(q6[r].abs(), k6[r].abs(), v6[r].abs(), a6[r], b6[r], s6.abs(), was[slot].abs())
        got = y[r].cpu().to(F64).reshape(n, heads, vd)
        assert bool(((got - o).abs() <= UNIT * oa + 1e-30).all()), (n, float(((got - o).abs() / oa).max()))
        assert bool(((now[slot] - S).abs() <= UNIT * Sa + 1e-30).all()), n
    st = st.cpu()
    assert torch.equal(st[0], whole[0]) and torch.equal(st[-1], whole[-1]) and torch.equal(st[:, :12], whole[:, :12])


def test_a_portion_goes_on_from_the_one_before():
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(4)
    heads, kd, vd, T = 2, 64, 64, 150
    x = torch.randn(T, heads * (2 * kd + vd), generator=g).to(DEV)
    q, k, v = x.split([heads * kd, heads * kd, heads * vd], 1)
    step = (torch.rand(T, heads, generator=g) * 0.1).to(DEV)
    decay = torch.exp(-4 * step)

    def run(cuts):
        state, out = torch.zeros(1, heads, kd, vd, device=DEV), []
        for lo, hi in zip(cuts, cuts[1:]):
            out.append(K.state_scan(q[lo:hi], k[lo:hi], v[lo:hi], step[lo:hi], decay[lo:hi], state, (None, i32([hi - lo]), i32([0]), i32([0])),
                                    heads, "additive", max_item_rows=1 if hi - lo == 1 else 0, chunks=True))
        return torch.cat(out), state

    y0, s0 = run([0, T])
    ya = K.state_scan(q.abs(), k.abs(), v.abs(), step, decay, torch.zeros(1, heads, kd, vd, device=DEV),
                      (None, i32([T]), i32([0]), i32([0])), heads, "additive")        # the sums of magnitudes
    for cuts in ([0, 1, 17, 64, 65, T], [0, 100, 101, T]):
        y, s = run(cuts)
        assert bool(((y - y0).abs() <= 2 * UNIT * ya + 1e-30).all()) and float((s - s0).norm() / s0.norm()) < 1e-6


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("what", ["q", "k", "v", "a", "b"])
def test_a_number_that_is_not_finite_reaches_no_row_before_it(what, bad):
    from swifttransformer_amd.ops import kernels as K
    heads, kd, vd, lens, at = 2, 64, 80, (130, 70), 130 + 25
    g = torch.Generator().manual_seed(8)
    T = sum(lens)
    items = (None, i32(list(lens)), i32([0, lens[0]]), i32([0, 1]))
    x = {n: torch.randn(T, heads * w, generator=g) for n, w in (("q", kd), ("k", kd), ("v", vd))}
    x["a"] = torch.rand(T, heads, generator=g) * 0.1
    x["b"] = torch.exp(-4 * x["a"])

    def run(y):
        state = torch.ones(2, heads, kd, vd, device=DEV)
        d = {n: t.to(DEV) for n, t in y.items()}
        out = K.state_scan(d["q"], d["k"], d["v"], d["a"], d["b"], state, items, heads, "additive", chunks=True)
        return out.view(T, heads, vd).cpu(), state.cpu()

    y0, s0 = run(x)
    spoilt = {n: t.clone() for n, t in x.items()}
    spoilt[what][at, 0 if what in "ab" else 5] = float("nan") if what == "b" else bad      # the first head of the second item's row 25
    y, s = run(spoilt)
    assert not bool((y[at, 0, 5] if what == "v" else y[at, 0]).isfinite().any())
    ok = torch.ones(T, heads, dtype=torch.bool)
    ok[at:, 0] = False
    # (a block that holds such a value is summed in another order: 16 products of weights and values up to 10 each)
    assert bool(((y - y0)[ok].abs() <= 16 * 2.0 ** -24 * 100).all())
    assert torch.equal(s[0], s0[0]) and torch.equal(s[1, 1], s0[1, 1])
    hit = s[1, 0, :, 5] if what == "v" else s[1, 0, 5] if what == "k" else s[1, 0]
    assert torch.equal(s, s0) if what == "q" else not bool(hit.isfinite().any())


@pytest.mark.parametrize("lens,heads,groups,kd,vd", [((2048,), 8, 1, 64, 64), ((700, 600, 33), 8, 2, 64, 128), ((33,), 16, 4, 64, 64),
                                                     ((130,), 16, 4, 64, 64), ((257, 77), 6, 6, 20, 36), ((300,), 4, 1, 128, 128), ((1,) * 48, 16, 4, 64, 64)])
def test_sums_are_no_further_from_float64_than_the_scans(monkeypatch, lens, heads, groups, kd, vd):
    """Against the kernel that goes row by row, on the same numbers."""
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + kd)
    T, B = sum(lens), len(lens)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    q, k, v = rnd(T, groups * kd), rnd(T, groups * kd), rnd(T, heads * vd)
    step = torch.rand(T, heads, generator=g, device=DEV) * 0.1 + 0.001
    decay = torch.exp(-(torch.rand(heads, generator=g, device=DEV) * 15 + 1) * step)
    skip, state = rnd(heads), rnd(B, heads, kd, vd)
    off = [sum(lens[:i]) for i in range(B)]
    items = (None, i32(list(lens)), i32(off), i32(list(range(B))))

    def run():
        s = state.clone()
        return K.state_scan(q, k, v, step, decay, s, items, heads, "additive", skip=skip, max_item_rows=1 if max(lens) == 1 else 0, chunks=True), s

    y, s = run()
    monkeypatch.setattr(K, "STATE_CHUNK_DIM", 0)
    y0, s0 = run()
    f = lambda t, n, w: t.to(F64).view(T, n, w).repeat_interleave(heads // n, 1)
    q6, k6, v6, a6, b6 = f(q, groups, kd), f(k, groups, kd), f(v, heads, vd), step.to(F64), decay.to(F64)
    want, last = torch.empty(T, heads, vd, dtype=F64, device=DEV), state.to(F64)
    for b in range(B):
        S = last[b]
        for t in range(off[b], off[b] + lens[b]):
            S = b6[t][:, None, None] * S + (a6[t][:, None] * k6[t])[:, :, None] * v6[t][:, None, :]
            want[t] = (S * q6[t][:, :, None]).sum(1) + skip.to(F64)[:, None] * v6[t]
        last[b] = S
    err = lambda x, z: float((x.to(F64).view(z.shape) - z).norm() / z.norm())
    # (prompts: 0.3 to 0.6 of the scan's; single rows 0.8, with the same state, whose one multiplication and addition are the scan's)
    assert err(y, want) <= err(y0, want), (err(y, want), err(y0, want))
    assert err(s, last) <= err(s0, last), (err(s, last), err(s0, last))


@pytest.mark.parametrize("lens,kd,vd", [((40, 1, 17), 64, 64), ((1, 16, 33, 130), 20, 100)])
def test_the_bound_on_an_items_rows_is_about_speed_alone(lens, kd, vd):
    """Items longer than the caller's bound come out as without one (the walk's sums and the scan's: the same products, 64 of them in
    another order)."""
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(kd)
    heads, T, B = 4, sum(lens), len(lens)
    x = torch.randn(T, heads * (2 * kd + vd), generator=g).to(DEV)
    q, k, v = x.split([heads * kd, heads * kd, heads * vd], 1)
    step = (torch.rand(T, heads, generator=g) * 0.1).to(DEV)
    decay, state = torch.exp(-4 * step), torch.randn(B, heads, kd, vd, generator=g).to(DEV)
    items = (None, i32(list(lens)), i32([sum(lens[:i]) for i in range(B)]), i32(list(range(B))[::-1]))

    def run(q, k, v, state, bound):
        s = state.clone()
        return K.state_scan(q, k, v, step, decay, s, items, heads, "additive", max_item_rows=bound), s

    (y, s), (y0, s0) = run(q, k, v, state, 1), run(q, k, v, state, 0)
    ya, sa = run(q.abs(), k.abs(), v.abs(), state.abs(), 0)                    # the sums of magnitudes
    assert bool(((y - y0).abs() <= 2 * UNIT * ya + 1e-30).all()) and bool(((s - s0).abs() <= 2 * UNIT * sa + 1e-30).all())
