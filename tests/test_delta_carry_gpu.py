"""The delta rule of many requests, whose chunks' states a workgroup carries 32 value channels at a time, against the same requests one by
one (16 channels a workgroup): the same sums in the same order, so the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# 384 (from 65 key channels on 256) / (heads * blocks of 32 value channels) requests with rows: one below, as many, and more
@pytest.mark.parametrize("heads,qk_heads,kd,vd,live", [(48, 16, 64, 32, 7), (48, 16, 64, 32, 8), (32, 8, 64, 64, 6), (32, 8, 64, 64, 9),
                                                       (40, 8, 16, 48, 5), (40, 8, 20, 48, 4), (32, 8, 128, 128, 1), (32, 8, 128, 128, 2),
                                                       (24, 6, 100, 100, 3), (32, 4, 7, 65, 70), (8, 4, 200, 40, 40)])
def test_many_requests_are_each_alone(heads, qk_heads, kd, vd, live):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator().manual_seed(heads + kd + live)
    taps, C = 4, 2 * qk_heads * kd + heads * vd
    lens = [(65, 1, 64, 130, 3, 17)[i % 6] if i < 12 else 1 + i % 3 for i in range(live)]
    T = sum(lens) + 1                                          # a row of no item
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    proj, taps_w, a_log, bias, gain = rnd(T, K.delta_row(heads, qk_heads, kd, vd)), rnd(taps, C) * 0.5, rnd(heads), rnd(heads), rnd(vd)
    was = rnd(live + 2, K.delta_slot(heads, qk_heads, kd, vd, taps))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    off = [sum(lens[:i]) for i in range(live)]
    token_item = i32([i for i, n in enumerate(lens) for _ in range(n)] + [-1])
    positions = i32([5 + p for n in lens for p in range(n)] + [-1])
    run = lambda x, state, ctx: K.delta_rule(x, taps_w, a_log, bias, gain, state, ctx, heads, qk_heads, kd, vd, 1e-5, 1e-6, torch.float32)
    together, alone = was.clone(), was.clone()
    # a list with room for more, and an entry of nobody between the requests
    at = [i if i < live // 2 else i + 1 for i in range(live)]
    il, of, sl = [0] * (live + 4), [0] * (live + 4), [-1] * (live + 4)
    for i, a in enumerate(at):
        il[a], of[a], sl[a] = lens[i], off[i], live - i
    where = torch.tensor(at + [-1], dtype=torch.int32, device=DEV)
    y = run(proj, together, (where[token_item.long()], positions, i32(il), i32(of), i32(sl)))
    for i, n in enumerate(lens):
        r = slice(off[i], off[i] + n)
        one = run(proj[r], alone, (i32([0] * n), positions[r].contiguous(), i32([n]), i32([0]), i32([live - i])))
        assert torch.equal(y[r], one), (i, n)
    assert torch.equal(together, alone) and torch.equal(alone[0], was[0]) and torch.equal(alone[-1], was[-1])
    assert bool(torch.isfinite(y[:-1]).all())
