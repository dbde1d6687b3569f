"""Partial results of attention with a sink, merged: every number of splits around the eight that are asked for at once, rows that end
within a workgroup's columns, heads whose columns four a thread do not divide, splits without keys; against float64.  And queries off
16-byte borders beside the same on them."""
import ctypes

import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("rows,heads,dim,splits", [(1, 1, 1, 1), (3, 5, 3, 2), (2, 32, 64, 7), (5, 32, 64, 8), (2, 20, 80, 9), (3, 100, 12, 16),
                                                   (1, 256, 32, 16), (200, 4, 64, 2), (2, 7, 130, 5)])
def test_merge(rows, heads, dim, splits):
    g = torch.Generator().manual_seed(rows + heads * splits)
    o = torch.randn(rows, splits, heads, dim, generator=g)
    m, l = torch.randn(rows, splits, heads, generator=g) * 3, torch.rand(rows, splits, heads, generator=g) + 0.1
    if splits > 1:                                  # a split without keys: no weight, whatever lies in its place
        m[:, -1], l[:, -1], o[:, -1] = float("-inf"), 0.0, float("nan")
    w = torch.exp(m.double() - m.double().amax(1, keepdim=True))
    want = (w[..., None] * o.double()).nan_to_num().sum(1) / (w * l.double()).sum(1)[..., None]
    ml = torch.stack([m, l], -1).to(DEV).contiguous()
    po, out = o.to(DEV).contiguous(), torch.empty(rows, heads * dim, device=DEV)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    K._check(K._lib().st_sink_attention_merge(ptr(out), ptr(po), ptr(ml), rows, heads, dim, splits, 0, ctypes.c_void_p(K._stream())))
    # float exponentials and up to 16 products a number: some 2^-24 each
    assert (out.cpu().double().view(want.shape) - want).abs().max().item() <= 32 * 2.0 ** -24 * want.abs().max().item()


@pytest.mark.parametrize("dtype,heads,kv,dk,dv,mixed", [(torch.bfloat16, 32, 8, 64, 64, True), (torch.bfloat16, 6, 3, 24, 40, True), (torch.float32, 8, 2, 20, 64, True),
                                                        (torch.bfloat16, 32, 32, 64, 128, False)])
def test_queries_off_their_borders(dtype, heads, kv, dk, dv, mixed):
    g = torch.Generator().manual_seed(3)
    rows, page, ctx = 5, 16, 150
    pages = -(-ctx // page)
    kc = torch.randn(pages, kv, page, dk, generator=g).to(dtype).to(DEV)
    vc = torch.randn(pages, kv, page, dv, generator=g).to(dtype).to(DEV)
    bt = torch.randperm(pages, generator=g).int().view(1, -1).to(DEV)
    item, pos = torch.zeros(rows, dtype=torch.int32, device=DEV), torch.tensor([0, 63, 64, 129, 149], dtype=torch.int32, device=DEV)
    q = torch.randn(rows, heads * dk, generator=g).to(dtype).to(DEV)
    wide = torch.zeros(rows, heads * dk + 9, dtype=dtype, device=DEV)
    wide[:, 1:1 + heads * dk] = q
    mix = torch.randn(heads * heads + 1, generator=g).to(DEV) * 0.1
    run = lambda x, m: K.sink_attention(x, kc, vc, item, pos, bt, heads, dk ** -0.5, head_mix=m, sink=True)
    m0, m1 = mix[1:].clone().view(heads, heads), mix[1:].view(heads, heads)
    assert torch.equal(run(q, m0 if mixed else None), run(wide[:, 1:1 + heads * dk], m1 if mixed else None))
