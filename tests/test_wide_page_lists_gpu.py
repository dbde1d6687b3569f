"""Page lists as wide as the row kernel of the attention has room for: it holds 16 numbers, a row of results a wave and the list."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,heads,kv_heads,hd,waves", [(torch.bfloat16, 4, 2, 64, 4), (torch.float32, 2, 2, 64, 8), (torch.bfloat16, 3, 1, 128, 8)])
def test_the_widest_list(dtype, heads, kv_heads, hd, waves):
    """The same numbers as with the list's used part alone (what lies behind it is not a page)."""
    g = torch.Generator(device="cuda").manual_seed(hd + waves)
    ps, lens = 16, [1, 70, 333]
    pages = [-(-n // ps) for n in lens]
    kc, vc = (torch.randn(sum(pages), kv_heads, ps, hd, generator=g, device="cuda").to(dtype) for _ in range(2))
    q = torch.randn(len(lens), heads * hd, generator=g, device="cuda").to(dtype)
    room = torch.cuda.get_device_properties(0).shared_memory_per_block // 4 - 16 - waves * hd
    used = max(pages)
    assert room > used
    table = torch.full((len(lens), room), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = torch.arange(at, at + n)
        at += n
    items, pos = torch.arange(len(lens), dtype=torch.int32, device="cuda"), torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
    run = lambda bt: K.attention_rows(q, kc, vc, items, pos, bt.cuda().contiguous(), heads, hd ** -0.5, num_waves=waves)
    wide, narrow = run(table), run(table[:, :used])
    torch.cuda.synchronize()
    assert torch.equal(wide, narrow) and bool(torch.isfinite(wide).all())
