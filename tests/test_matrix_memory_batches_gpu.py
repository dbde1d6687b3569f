"""Single tokens through the matrix memory: a thread has one to eight pieces of the state at a time, by the numbers of key and value
channels; against float64, from a state that is not empty."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# pieces a thread: 1 (fewer pieces than threads), 2, 2 (the last one past the keys), 4, 4 (of a row that does not fill the waves), 7, 16 in two batches
@pytest.mark.parametrize("heads,dk,dv", [(2, 8, 16), (1, 64, 128), (3, 60, 128), (2, 128, 128), (1, 96, 132), (1, 100, 256), (2, 256, 256)])
def test_one_token_from_a_state(heads, dk, dv):
    g = torch.Generator().manual_seed(heads * 1000 + dk + dv)
    rnd = lambda *s: torch.randn(*s, generator=g)
    cap, eps = 12.0, 1e-5
    q, k, v, gate = rnd(heads, dk), rnd(heads, dk), rnd(heads, dv), rnd(heads, dv)
    zi, zf, bi, bf, gain = rnd(heads), rnd(heads), rnd(heads), rnd(heads), 1 + 0.2 * rnd(heads * dv)
    S, n, m = rnd(heads, dk, dv), rnd(heads, dk), rnd(heads)
    state = torch.full((3, K.memory_slot(heads, dk, dv)), 5.0)
    state[1, :heads * (dk * dv + dk + 1)] = torch.cat([S.flatten(), n.flatten(), m])
    state = state.to(DEV)
    proj = torch.cat([t.flatten() for t in (q, k, v, gate, zi, zf)])[None].to(DEV)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    out = K.matrix_memory(proj, bi.to(DEV), bf.to(DEV), gain.to(DEV), state, (i32(0), i32(1), i32(0), i32(1)), heads, dk, dv, cap, eps, torch.float32,
                          all_single=True)
    d = lambda t: t.double()
    i = cap * torch.tanh(d(zi + bi) / cap)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh(d(zf + bf) / cap))
    m_new = torch.maximum(f + d(m), i)
    keep, add = (f + d(m) - m_new).exp(), (i - m_new).exp()
    S_new = keep[:, None, None] * d(S) + add[:, None, None] * d(k)[:, :, None] * d(v)[:, None, :]
    n_new = keep[:, None] * d(n) + add[:, None] * d(k)
    qs = d(q) * dk ** -0.5
    den = torch.maximum((n_new * qs).sum(1).abs(), (-m_new).exp()) + 1e-6
    o = (S_new * qs[:, :, None]).sum(1) / den[:, None]
    want = o / (o.square().mean(1, keepdim=True) + eps).sqrt() * d(gain).view(heads, dv) * torch.sigmoid(d(gate))
    # float sums of up to 256 products, and the norm's: some roundings of 2^-24 of the largest
    assert (out[0].cpu().double() - want.flatten()).abs().max() <= 2e-6 * want.abs().max()
    got = state.cpu().double()
    assert (got[1, :heads * dk * dv].view(heads, dk, dv) - S_new).abs().max() <= 1e-6 * S_new.abs().max()
    assert (got[1, heads * dk * dv:heads * (dk * dv + dk)].view(heads, dk) - n_new).abs().max() <= 1e-6 * n_new.abs().max()
    assert (got[1, heads * (dk * dv + dk):heads * (dk * dv + dk + 1)] - m_new).abs().max() <= 1e-6 * (1 + m_new.abs().max())
    assert (got[[0, 2]] == 5.0).all()
