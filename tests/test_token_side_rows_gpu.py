"""The token side input of many bfloat16 rows (two a workgroup) against float64.

Bound: the gate's sums have at most ``width`` / 256 + 20 roundings of 2^-24 in a chain, GELU and the projection two dozen more, and the unit
norm divides by a length that moves by as much: relative to the projection's own length, 2^-24 (width / 256 + 64), times what GELU makes of an
error in its argument (at most 1.13 of it, in the size of the products that are summed)."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


# around the lines of the rule (256 rows, two workgroups a unit) and of the columns a thread (1,024, 2,048), odd rows, both sizes of the gate
@pytest.mark.parametrize("rows,width,dim", [(257, 768, 16), (300, 1000, 8), (511, 1024, 16), (512, 1032, 16), (513, 2048, 16), (1023, 2048, 8),
                                            (600, 2560, 16), (259, 4096, 16), (1100, 64, 16)])
def test_many_rows(rows, width, dim):
    g = torch.Generator(device="cuda").manual_seed(rows + width + dim)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, vocab = rand(rows, width), 50
    ids = torch.randint(0, vocab, (rows,), generator=g, device="cuda", dtype=torch.int32)
    item = torch.zeros(rows, dtype=torch.int32, device="cuda")
    item[rows - 3], item[5] = -1, -1                    # padding rows
    ids[rows - 1], ids[8] = -1, vocab                   # tokens outside the table: nothing is added
    whole = rand(vocab, 3 * dim).bfloat16()
    table, wg, wp, gain = whole[:, dim:2 * dim], (rand(dim, width) * 0.05).bfloat16(), (rand(width, dim) * 0.05).bfloat16(), rand(width)
    got = K.token_side(x.clone(), ids, item, table, wg, wp, gain, 1e-5)
    z = x.double() @ wg.double().T
    known = (ids >= 0) & (ids < vocab)
    e = torch.where(known[:, None], table[ids.clamp(0, vocab - 1).long()].double(), 0.0)
    h = 0.5 * z * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (z + 0.044715 * z ** 3))) * e
    y = h @ wp.double().T
    length = torch.sqrt(y.square().mean(1, keepdim=True) + 1e-5)
    add = y / length * gain.double()
    add[item < 0] = 0.0
    size = (x.double().abs() @ wg.double().abs().T) * 1.13 * e.abs()         # of the sums behind a gated number
    off = 2.0 ** -24 * (width / 256 + 64) * (size @ wp.double().abs().T / length + add.abs())
    off = off + 2.0 ** -24 * (width / 256 + 64) * size.sum(1, keepdim=True) * wp.double().abs().max() / length * gain.double().abs()
    want = x.double() + add
    assert bool(((got.double() - want).abs() <= off * gain.double().abs().clamp(min=1) + 2.0 ** -22 * want.abs()).all())
    assert torch.equal(got[item < 0], x[item < 0])
    assert torch.equal(got[~known], x[~known])


def test_same_as_a_row_a_workgroup():
    """256 rows go a row a workgroup: the same rows among more of them, to float's rounding."""
    g = torch.Generator(device="cuda").manual_seed(2)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, ids = rand(700, 2048), torch.randint(0, 90, (700,), generator=g, device="cuda", dtype=torch.int32)
    item = torch.zeros(700, dtype=torch.int32, device="cuda")
    table, wg, wp, gain = rand(90, 16).bfloat16(), (rand(16, 2048) * 0.05).bfloat16(), (rand(2048, 16) * 0.05).bfloat16(), rand(2048)
    many = K.token_side(x.clone(), ids, item, table, wg, wp, gain, 1e-5)
    for a in range(0, 700, 250):
        b = min(700, a + 250)
        few = K.token_side(x[a:b].clone(), ids[a:b].contiguous(), item[a:b].contiguous(), table, wg, wp, gain, 1e-5)
        assert float((many[a:b] - few).abs().max()) <= 1e-4
