"""Gated linear attention by chunks against the recurrence in float64: items of 1 row to several chunks around the limits of a block (16),
of a walk (16) and of a chunk (64), sizes with and without whole 16-byte pieces, decays of exactly 0 and 1, padding items, and a
portion that goes on from the state another one left."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


def _walk(q, k, v, a, S):
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=F64)
    for t in range(q.shape[0]):
        S = a[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out[t] = (S * q[t][:, :, None]).sum(1)
    return out, S


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,heads,kd,vd", [((1, 15, 16, 17, 63), 3, 64, 64), ((64, 65, 1, 129), 2, 128, 128), ((200, 2), 2, 5, 7),
                                              ((33, 80, 3), 3, 80, 48), ((130,), 2, 20, 100), ((1,) * 70, 2, 64, 32),
                                              ((70,) + (1,) * 66, 1, 16, 16)])
def test_chunks_are_the_recurrence(dtype, lens, heads, kd, vd):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(sum(lens) + kd)
    T, B = sum(lens) + 2, len(lens) + 1                        # two rows of no item; one padding item
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype)
    proj = rnd(T, heads * (2 * kd + 2 * vd) + (3 if kd == 5 else 0))
    logits = torch.randn(T, heads * kd, generator=g) * 3
    logits[::7, ::3] = -1e5                                    # decays of exactly 0 and 1
    logits[::5, 1::3] = 1e5
    logits[9, :] = -1e5
    a = torch.sigmoid(logits.to(F64)) ** 0.25
    state = torch.randn(B + 2, heads, kd, vd, generator=g)
    gain = torch.rand(vd, generator=g) + 0.5
    eps, scale = 1e-5, kd ** -0.5
    off = [sum(lens[:i]) for i in range(len(lens))]
    slots = list(range(len(lens), 0, -1))                      # slot 0 and the last stay untouched
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    items = (None, i32(list(lens) + [0]), i32(off + [0]), i32(slots + [-1]))
    d = proj.to(DEV)
    cut = [heads * kd, 2 * heads * kd, 2 * heads * kd + heads * vd, 2 * heads * (kd + vd)]
    q, k, v, gate = (d[:, lo:hi] for lo, hi in zip([0] + cut, cut))
    st = state.to(DEV)
    y = K.gla_chunks(q, k, v, logits.to(DEV), 4.0, st, items, heads, scale, gate, gain.to(DEV), eps, single=max(lens) == 1)
    # the roundings on a number's way: up to 16 + 4 + 32 decays of a few each, 64 + 128 products and sums in chains of fours; in units
    # of 2^-24 of the sum of magnitudes
    unit = 512 * 2.0 ** -24
    f = lambda x, w: x.cpu().to(F64).reshape(T, heads, w)
    q6, k6, v6, a6, g6 = f(q, kd) * scale, f(k, kd), f(v, vd), a.to(F64).reshape(T, heads, kd), f(gate, vd)
    for n, lo, slot in zip(lens, off, slots):
        r = slice(lo, lo + n)
        o, S = _walk(q6[r], k6[r], v6[r], a6[r], state[slot].to(F64))
        oa, Sa = _walk(q6[r].abs(), k6[r].abs(), v6[r].abs(), a6[r], state[slot].to(F64).abs())
        rms = torch.sqrt(o.square().mean(-1, keepdim=True) + eps)
        b = unit * oa
        by = gain.to(F64) * (g6[r] * torch.sigmoid(g6[r]))
        want = o / rms * by
        err_rms = b.square().mean(-1, keepdim=True).sqrt() / rms
        bound = by.abs() * (b / rms + o.abs() / rms * err_rms) + (2.0 ** -8 if dtype == torch.bfloat16 else 1e-6) * want.abs() + 1e-12
        got = y[r].cpu().to(F64).reshape(n, heads, vd)
        assert bool(((got - want).abs() <= bound).all()), (n, float(((got - want).abs() / bound).max()))
        assert bool(((st[slot].cpu().to(F64) - S).abs() <= unit * Sa + 1e-12).all()), n
    assert torch.equal(st[0].cpu(), state[0]) and torch.equal(st[-1].cpu(), state[-1])


def test_a_portion_goes_on_from_the_one_before():
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(4)
    heads, kd, vd, T = 2, 64, 64, 150
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    x = torch.randn(T, 2 * heads * (kd + vd), generator=g).to(DEV)
    q, k, v, gate = x.split([heads * kd, heads * kd, heads * vd, heads * vd], 1)
    z = torch.randn(T, heads * kd, generator=g).to(DEV)
    gain = torch.ones(vd, device=DEV)

    def run(cuts):
        state = torch.zeros(1, heads, kd, vd, device=DEV)
        out = []
        for lo, hi in zip(cuts, cuts[1:]):
            items = (None, i32([hi - lo]), i32([0]), i32([0]))
            out.append(K.gla_chunks(q[lo:hi], k[lo:hi], v[lo:hi], z[lo:hi].contiguous(), 8.0, state, items, heads, 0.125, gate[lo:hi], gain, 1e-5,
                                    single=hi - lo == 1))
        return torch.cat(out), state

    y0, s0 = run([0, T])
    for cuts in ([0, 1, 17, 64, 65, T], [0, 100, 101, T]):
        y, s = run(cuts)
        # float sums in another order (see above: 256 roundings), of numbers up to 5 after the norm
        assert float((y - y0).abs().max()) < 256 * 2.0 ** -24 * 5 * 8 and float((s - s0).norm() / s0.norm()) < 1e-6


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("what", ["q", "k", "v", "z"])
def test_a_number_that_is_not_finite_reaches_no_row_before_it(what, bad):
    from swifttransformer_amd.ops import kernels as K
    heads, kd, vd, lens, at = 2, 64, 48, (130, 70), 130 + 25
    g = torch.Generator().manual_seed(8)
    T = sum(lens)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    items = (None, i32(list(lens)), i32([0, lens[0]]), i32([0, 1]))
    x = {n: torch.randn(T, heads * w, generator=g) for n, w in (("q", kd), ("k", kd), ("v", vd), ("z", kd), ("g", vd))}

    def run(y):
        state = torch.ones(2, heads, kd, vd, device=DEV)
        d = {n: t.to(DEV) for n, t in y.items()}
        out = K.gla_chunks(d["q"], d["k"], d["v"], d["z"], 8.0, state, items, heads, 0.125, d["g"], torch.ones(vd, device=DEV), 1e-5)
        return out.view(T, heads, vd).cpu(), state.cpu()

    y0, s0 = run(x)
    spoilt = {n: t.clone() for n, t in x.items()}
    spoilt[what][at, 5] = float("nan") if what == "z" else bad            # the first head of the second item's row 25
    y, s = run(spoilt)
    assert not bool(y[at, 0].isfinite().all())                             # (an infinite root mean square makes the other channels zero)
    ok = torch.ones(T, heads, dtype=torch.bool)
    ok[at:, 0] = False
    # (a block that holds such a value is summed in another order: 16 products, of numbers up to 50 after the norm)
    assert bool(((y - y0)[ok].abs() <= 16 * 2.0 ** -24 * 50).all())
    assert torch.equal(s[0], s0[0]) and torch.equal(s[1, 1], s0[1, 1])
    hit = s[1, 0] if what == "q" else s[1, 0, :, 5] if what == "v" else s[1, 0, 5]
    assert torch.equal(s[1, 0], s0[1, 0]) if what == "q" else not bool(hit.isfinite().any())


@pytest.mark.parametrize("lens,heads,kd,vd,tau", [((2011,), 8, 64, 64, 16.0), ((700, 600, 33), 8, 64, 128, 16.0), ((17,), 16, 64, 64, 4.0),
                                                  ((33,), 16, 64, 64, 1.0), ((130,), 16, 64, 64, 1.0), ((257, 77), 6, 20, 36, 16.0),
                                                  ((300,), 4, 128, 128, 16.0), ((1,) * 48, 16, 64, 64, 1.0), ((1,) * 24, 8, 128, 128, 16.0),
                                                  ((16, 9, 2), 8, 128, 128, 16.0), ((500,), 16, 64, 64, 0.25)])
def test_sums_are_no_further_from_float64_than_the_scans(lens, heads, kd, vd, tau):
    """Against decay gates, the kernel that goes row by row, and the norm behind it, on the same numbers."""
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + kd)
    T, B = sum(lens), len(lens)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    q, k, v, gate, z = rnd(T, heads * kd), rnd(T, heads * kd), rnd(T, heads * vd), rnd(T, heads * vd), rnd(T, heads * kd) * 2
    state, gain, eps, scale = rnd(B, heads, kd, vd), torch.ones(vd, device=DEV), 1e-5, kd ** -0.5
    off = [sum(lens[:i]) for i in range(B)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    items, single = (None, i32(list(lens)), i32(off), i32(list(range(B)))), max(lens) == 1
    s, s0 = state.clone(), state.clone()
    y = K.gla_chunks(q, k, v, z, tau, s, items, heads, scale, gate, gain, eps, single=single)
    o = K.gla_scan(q, k, v, K.decay_gate(z.clone(), 1.0 / tau), s0, items, heads, scale, 16 if single else 8)
    y0 = K.gated_head_norm(o, gate, gain, heads, eps, torch.float32)
    f = lambda t, w: t.to(F64).view(T, heads, w)
    q6, k6, v6, g6, a6 = f(q, kd) * scale, f(k, kd), f(v, vd), f(gate, vd), torch.sigmoid(f(z, kd)) ** (1.0 / tau)
    want, last = torch.empty(T, heads, vd, dtype=F64, device=DEV), state.to(F64)
    for b in range(B):
        S = last[b]
        for t in range(off[b], off[b] + lens[b]):
            S = a6[t][:, :, None] * S + k6[t][:, :, None] * v6[t][:, None, :]
            want[t] = (S * q6[t][:, :, None]).sum(1)
        last[b] = S
    want = want * torch.rsqrt(want.square().mean(-1, keepdim=True) + eps) * (g6 * torch.sigmoid(g6))
    err = lambda x, w: float((x.to(F64).view(w.shape) - w).norm() / w.norm())
    assert err(y, want) <= err(y0, want), (err(y, want), err(y0, want))
    assert err(s, last) <= err(s0, last), (err(s, last), err(s0, last))


@pytest.mark.parametrize("lens,kd,vd", [((40, 1, 17), 64, 64), ((1, 16, 33, 130), 20, 100), ((50,), 128, 128)])
def test_items_of_a_step_said_to_be_single_may_be_longer(lens, kd, vd):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(kd)
    heads, T, B = 3, sum(lens), len(lens)
    q, k, v, gate, z = (torch.randn(T, heads * w, generator=g).to(DEV) for w in (kd, kd, vd, vd, kd))
    state, gain = torch.randn(B, heads, kd, vd, generator=g).to(DEV), torch.ones(vd, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    items = (None, i32(list(lens)), i32([sum(lens[:i]) for i in range(B)]), i32(list(range(B))[::-1]))

    def run(single):
        s = state.clone()
        return K.gla_chunks(q, k, v, z, 4.0, s, items, heads, kd ** -0.5, gate, gain, 1e-5, single=single), s

    (y, s), (y0, s0) = run(True), run(False)
    # (the same float sums in another order: 256 roundings, of numbers up to 5 after the norm and 5 of the gate)
    assert float((y - y0).abs().max()) < 256 * 2.0 ** -24 * 5 * 8 and float((s - s0).norm() / s0.norm()) < 1e-6
