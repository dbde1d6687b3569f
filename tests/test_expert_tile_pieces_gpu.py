"""Experts' tiles of 128 places by 256 weight rows: what whole rounds of a die's compute units leave over goes in halves or quarters of a
tile.  Numbers of tiles and of blocks that leave one, a few, a quarter, half and more than half of a round, blocks and tiles that end
early; the inputs' and the output's product against float64."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# pairs of each of four experts, features, depth (tiles x blocks of 128 or 256 features over eight dies of 32 units)
UP = [((630, 640, 513, 640), 1664, 72),        # 260 items: 33 a die, one left over; 29 on the last
      ((630, 640, 513, 520), 2048, 136),       # 320: 8 left over
      ((760, 641, 700, 645), 2048, 64),        # 384: 16 left over
      ((630, 640, 600, 640), 2052, 200),       # 340: 11 left over, 7 on the last; the last block has four features
      ((300, 300, 0, 300), 2560, 64),          # 180: 23, no whole round and more than half of one
      ((1, 1280, 0, 129), 2176, 128)]          # an expert of one pair; 221 items


@pytest.mark.parametrize("counts,features,depth", UP)
@pytest.mark.parametrize("kind", ["gated", "gelu", "output"])
def test_pieces(counts, features, depth, kind):
    lib, ptr = K._lib(), K._ptr
    E, pairs = len(counts), sum(counts)
    if kind == "output":
        features *= 2                           # blocks of 256 features
    g = torch.Generator(device=DEV).manual_seed(pairs + features)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=DEV) * std).bfloat16()
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(pairs, generator=torch.Generator().manual_seed(1))].int().to(DEV)
    cap = K.moe_capacity(pairs, 1, E, 128)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device=DEV)
    srt, place, expert = i32(cap), i32(pairs), i32(cap // 128)
    K._check(lib.st_moe_align(ptr(srt), ptr(place), ptr(expert), ptr(ids), pairs, E, cap, 128, K._stream()))
    w, w2 = rnd(E, features, depth, std=depth ** -0.5), rnd(E, features, depth, std=depth ** -0.5)
    at = place.long()
    if kind == "output":
        y, out = rnd(cap, depth), torch.full((cap, features), float("nan"), device=DEV)
        K._check(lib.st_moe_down(None, None, ptr(out), ptr(y), ptr(w), ptr(srt), ptr(expert), cap, 128, 2, features, depth, 1.0, 1, K._stream()))
        got, want = out[at].double(), torch.stack([w[e].double() @ v for e, v in zip(ids.long().tolist(), y[at].double())])
        assert out[(srt < 0).nonzero()[:, 0]].isnan().all()              # places without a pair stay
        assert (got - want).abs().max().item() <= 4e-7 * depth ** 0.5 * 8    # exact products of size one, summed in float
        return
    x, y = rnd(pairs, depth), rnd(cap, features)
    weights = torch.rand(pairs, generator=g, device=DEV)
    gated = kind == "gated"
    K._check(lib.st_moe_up(ptr(y), ptr(x), ptr(w) if gated else None, ptr(w2), ptr(srt), ptr(expert), ptr(weights), cap, 128, 1, depth, features, 7.0, 1 if gated else 2,
                           1, K._stream()))
    xd = x.double()
    u = torch.empty(pairs, features, dtype=torch.float64, device=DEV)
    gate = torch.empty_like(u)
    for e in range(E):
        rows = (ids == e).nonzero()[:, 0]
        u[rows], gate[rows] = xd[rows] @ w2[e].double().T, xd[rows] @ w[e].double().T
    want = gate * torch.sigmoid(gate) * u if gated else torch.nn.functional.gelu(u)
    got = y[at].double()
    # bfloat16 results: half of 2^-8 of each, and the products' float sums
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 4e-7 * depth ** 0.5 * 20).all()
