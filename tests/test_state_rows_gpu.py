"""Single tokens through the additive recurrence (a row's operands and state asked for at once): the numbers of the walk over several rows."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("items,heads,qk,dk,dv", [(1, 4, 4, 64, 128), (9, 6, 3, 64, 64), (5, 4, 2, 20, 72), (40, 2, 2, 8, 24), (3, 5, 5, 61, 100)])
def test_two_steps_are_one_walk(items, heads, qk, dk, dv):
    g = torch.Generator(device="cuda").manual_seed(items + dk)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q, k, v = rnd(2 * items, qk * dk), rnd(2 * items, qk * dk), rnd(2 * items, heads * dv)
    a, b = rnd(2 * items, heads), torch.rand(2 * items, heads, generator=g, device="cuda") * 0.2 + 0.8
    start = rnd(items + 1, heads, dk, dv)
    slots = list(range(items))[::-1]
    slots[items // 2] = -1                               # an item without a slot is left alone
    walked = start.clone()
    both = K.state_scan(q, k, v, a, b, walked, (i32([i // 2 for i in range(2 * items)]), i32([2] * items), i32([2 * i for i in range(items)]), i32(slots)),
                        heads, "additive", max_item_rows=1)
    stepped = start.clone()
    for r in range(2):
        rows = torch.arange(items, device="cuda") * 2 + r
        one = K.state_scan(q[rows], k[rows], v[rows], a[rows], b[rows], stepped,
                           (i32(list(range(items))), i32([1] * items), i32(list(range(items))), i32(slots)), heads, "additive", max_item_rows=1)
        live = [i for i in range(items) if slots[i] >= 0]
        assert torch.equal(one.view(items, -1)[live], both.view(2 * items, -1)[rows[live]])
    assert torch.equal(stepped, walked) and torch.equal(stepped[items], start[items])
