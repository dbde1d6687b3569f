"""Single tokens of many requests through the delta rule (workgroups of 512 threads, eight pieces of state each) against float64.

Bound: S^T k and S^T q are sums of ``dk`` products in float, dk roundings of 2^-24 of the sum of absolute values at most; the unit lengths, the
gates and SiLU add some 40 more, and the output's norm divides by a length that moves by as much."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("items,heads,qk,dk,dv,taps", [(9, 32, 8, 128, 128, 4), (65, 4, 4, 128, 128, 1), (24, 12, 3, 100, 96, 3), (9, 32, 8, 64, 256, 4),
                                                       (40, 8, 8, 68, 240, 2), (9, 32, 16, 256, 256, 4),
                                                       (32, 32, 8, 64, 128, 4), (33, 32, 8, 64, 128, 4)])   # (either side of four workgroups a unit)
def test_many_requests(items, heads, qk, dk, dv, taps):
    g = torch.Generator(device="cuda").manual_seed(items + dk + dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    C = 2 * qk * dk + heads * dv
    proj, w, a_log, bias, gain = rnd(items, K.delta_row(heads, qk, dk, dv)), rnd(taps, C) * 0.5, rnd(heads) * 0.3, rnd(heads), rnd(dv)
    state = rnd(items + 1, K.delta_slot(heads, qk, dk, dv, taps))
    was = state.clone()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    slots = torch.randperm(items, generator=torch.Generator().manual_seed(1)).int().cuda()
    pos = i32([7] * items)
    ctx = (torch.arange(items, dtype=torch.int32, device="cuda"), pos, i32([1] * items), torch.arange(items, dtype=torch.int32, device="cuda"), slots)
    out = K.delta_rule(proj, w, a_log, bias, gain, state, ctx, heads, qk, dk, dv, 1e-5, 1e-6, torch.float32, all_single=True)
    assert torch.equal(state[items], was[items])
    # the formula; a slot's last inputs lie by position modulo the taps, then the states
    base, P = (taps * C + 3) // 4 * 4, proj.double()
    ring = was[slots.long(), :taps * C].view(items, taps, C).double()
    S = was[slots.long(), base:base + heads * dk * dv].view(items, heads, dk, dv).double()
    f = w[taps - 1].double() * P[:, :C]
    for j in range(1, taps):
        f = f + w[taps - 1 - j].double() * ring[:, (7 - j) % taps]
    f = f * torch.sigmoid(f)
    q, k, v = f[:, :qk * dk].view(items, qk, dk), f[:, qk * dk:2 * qk * dk].view(items, qk, dk), f[:, 2 * qk * dk:].view(items, heads, dv)
    unit = lambda y: (y / torch.sqrt(y.square().sum(-1, keepdim=True) + 1e-6)).repeat_interleave(heads // qk, 1)
    q, k = unit(q) * dk ** -0.5, unit(k)
    z, b, a = P[:, C:C + heads * dv].view(items, heads, dv), P[:, C + heads * dv:C + heads * dv + heads], P[:, C + heads * dv + heads:C + heads * dv + 2 * heads]
    decay = torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(a + bias.double()))[..., None]
    u = torch.sigmoid(b)[..., None] * (v - decay * (S * k[..., None]).sum(2))
    new = decay[..., None] * S + k[..., None] * u[:, :, None]
    o = (new * q[..., None]).sum(2)
    eps = 2.0 ** -24 * (dk + 40)
    size_u = v.abs() + decay * (S.abs() * k.abs()[..., None]).sum(2)
    got = state[slots.long(), base:base + heads * dk * dv].view(items, heads, dk, dv).double()
    assert bool(((got - new).abs() <= eps * (decay[..., None] * S.abs() + 2 * k.abs()[..., None] * size_u[:, :, None])).all())
    length = torch.sqrt(o.square().mean(-1, keepdim=True) + 1e-5)
    size_o = ((decay[..., None] * S.abs() + 2 * k.abs()[..., None] * size_u[:, :, None]) * q.abs()[..., None]).sum(2)
    y = o / length * gain.double() * z * torch.sigmoid(z)
    near = (size_o + o.abs() / length * torch.sqrt(size_o.square().mean(-1, keepdim=True))) / length
    assert bool(((out.view(items, heads, dv).double() - y).abs() <= 2 * eps * near * (gain.double() * z * torch.sigmoid(z)).abs() + 1e-9).all())
