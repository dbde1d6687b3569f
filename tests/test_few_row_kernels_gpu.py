"""Elementwise kernels that few rows go through in smaller pieces: the same numbers, to the last bit, as among many rows."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


# either side of 256 numbers a compute unit (256 units: 65,536), widths of whole pieces of 16 bytes and others
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [1024, 1000, 1003])
@pytest.mark.parametrize("kind", ["gelu_tanh", "silu", "relu_squared", "none"])
def test_activation_multiply(dtype, width, kind):
    g = torch.Generator(device="cuda").manual_seed(width)
    ab = torch.randn(200, 2 * width, generator=g, device="cuda").to(dtype)
    a, b = ab[:, :width], ab[:, width:]
    many, alone = K.activation_multiply(a, b, kind), K.activation_multiply(a, None, kind)
    for lo, hi in ((0, 1), (1, 65), (65, 129), (129, 194)):
        assert torch.equal(K.activation_multiply(a[lo:hi], b[lo:hi], kind), many[lo:hi])
        assert torch.equal(K.activation_multiply(a[lo:hi], None, kind), alone[lo:hi])


@pytest.mark.parametrize("W,E,top,identity", [(2048, 9, 3, 0), (72, 6, 2, 2), (5000, 5, 2, 0), (1023, 9, 4, 0)])
def test_sums_of_experts(W, E, top, identity):
    """As many tokens as units are summed by more threads each than more tokens are."""
    g = torch.Generator(device="cuda").manual_seed(W)
    T = 700
    po, place = torch.randn(T * top, W, generator=g, device="cuda"), torch.randperm(T * top, generator=g, device="cuda").int()
    wts = torch.rand(T * top, generator=g, device="cuda")
    ids = torch.randint(0, E + identity, (T * top,), generator=g, device="cuda").int()
    place[ids >= E] = -1
    x, res = torch.randn(T, W, generator=g, device="cuda").bfloat16(), torch.randn(T, W, generator=g, device="cuda")
    p = lambda t: t.data_ptr() if t is not None else None

    def run(lo, hi):
        out = torch.empty(hi - lo, W, device="cuda")
        parts = [t[lo * top:hi * top].contiguous() for t in (place, wts, ids)]
        rows = [t[lo:hi].contiguous() for t in (res, x)]
        assert K._lib().st_moe_combine(p(out), p(rows[0]), p(po), p(parts[0]), p(parts[1]), p(parts[2]), p(rows[1]) if identity else None, E, hi - lo, top, W,
                                       0.5, 1, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out
    many = run(0, T)
    for lo, hi in ((0, 1), (1, 100), (100, 356)):
        assert torch.equal(run(lo, hi), many[lo:hi])
