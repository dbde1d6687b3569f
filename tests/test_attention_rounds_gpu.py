"""Decode attention where its rounds of keys end: contexts around one, two and three rounds of a workgroup's groups, page sizes that no
shift divides by, heads that do not fill their lanes; against float64, with NaN in every cache entry that no query sees."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype,head_dim,page", [(torch.bfloat16, 64, 16), (torch.bfloat16, 80, 12), (torch.bfloat16, 128, 1),
                                                 (torch.bfloat16, 16, 7), (torch.float32, 64, 16), (torch.float32, 48, 3)])
def test_rounds(dtype, head_dim, page, waves):
    lanes = 1
    while lanes * (8 if dtype == torch.bfloat16 else 4) < head_dim:
        lanes *= 2
    a_round = waves * (64 // lanes) * 4
    lens = sorted({1, 2, a_round // 4, a_round - 1, a_round, a_round + 1, 2 * a_round - 1, 2 * a_round, 2 * a_round + 1,
                   3 * a_round - 1, 3 * a_round + 1, 4 * a_round + 5})
    rows, heads, kv = len(lens), 4, 2
    pages = -(-max(lens) // page)
    g = torch.Generator().manual_seed(7)
    k, v = (torch.full((rows * pages + 1, kv, page, head_dim), float("nan")) for _ in range(2))
    table = torch.randperm(rows * pages, generator=g).int().view(rows, pages)
    q = torch.randn(rows, heads * head_dim, generator=g).to(dtype)
    want = torch.empty(rows, heads * head_dim, dtype=torch.float64)
    scale = head_dim ** -0.5
    for r, n in enumerate(lens):
        kk, vv = (torch.randn(n, kv, head_dim, generator=g).to(dtype) for _ in range(2))
        for j in range(n):
            k[table[r, j // page], :, j % page] = kk[j].float()
            v[table[r, j // page], :, j % page] = vv[j].float()
        for h in range(heads):
            s = kk[:, h // 2].double() @ q[r, h * head_dim:(h + 1) * head_dim].double() * scale
            want[r, h * head_dim:(h + 1) * head_dim] = torch.softmax(s, 0) @ vv[:, h // 2].double()
    put = lambda t: t.to(DEV)
    items, positions = torch.arange(rows).int(), torch.tensor(lens).int() - 1
    got = K.attention_rows(put(q), put(k.to(dtype)), put(v.to(dtype)), put(items), put(positions), put(table), heads, scale,
                           num_waves=waves).cpu().double()
    # bfloat16: the result is rounded to it (2^-9 of itself) and the exponential is the hardware's; float: sums of up to some hundred
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 1e-5
    assert (got - want).abs().max().item() <= tol * want.abs().max().item()
