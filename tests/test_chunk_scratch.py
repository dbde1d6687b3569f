"""Room for the states of the chunked recurrences: one a chunk of 64 rows, and one more for each item that may have more than 16 rows."""
import random

import pytest
import torch

from swifttransformer_amd.ops import kernels as K


def test_the_count_is_enough_and_no_more_than_one_an_item():
    rng = random.Random(5)
    for _ in range(2000):
        lens = [rng.choice((0, 1, 1, 16, 17, 18, 63, 64, 65, rng.randint(1, 300))) for _ in range(rng.randint(1, 40))]
        rows = sum(lens) + rng.choice((0, 0, 3))
        n = K._chunk_states(rows, len(lens))
        assert sum(-(-x // 64) for x in lens if x > 16) <= n <= rows // 64 + len(lens)
    assert K._chunk_states(256, 256) == 4 + 15 and K._chunk_states(16, 16) == 0 and K._chunk_states(2048, 1) == 33


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["gla", "state"])
def test_requests_of_single_tokens_want_no_room(what):
    """240 single tokens beside a portion of 33: room for a few states and not for 240."""
    heads, d, singles = 4, 64, 240
    B, T = singles + 1, singles + 33
    dev = "cuda"
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    items = (None, i32([1] * singles + [33]), i32(list(range(B))), i32(list(range(B))))
    x = [torch.randn(T, heads * d, device=dev) for _ in range(5)]
    state, gain, gates = torch.zeros(B, heads, d, d, device=dev), torch.ones(d, device=dev), torch.rand(T, heads, device=dev)

    def run():
        if what == "gla":
            return K.gla_chunks(x[0], x[1], x[2], x[3], 4.0, state, items, heads, 0.125, x[4], gain, 1e-5)
        return K.state_scan(x[0], x[1], x[2], gates, gates, state, items, heads, "additive", chunks=True)

    run()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    run()
    one = 4 * heads * d * (d + 1)
    assert torch.cuda.max_memory_allocated() - before <= 4 * T * heads * d + (T // 64 + T // 17) * one + (1 << 20)
