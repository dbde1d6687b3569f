"""The few-row product at the edges of its slabs: depths that end within a step, within a wave's share or before a wave's first step,
features that end within a tile of 8, 16, 24 or 32, every number of rows, operands the epilogue cannot take 16 bytes of; against float64."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def draw(seed, *shape, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(DEV)


def close(got, want, x, w, added):
    """Products of bfloat16 numbers are exact in float; sums of `depth` of them in float, in some order, are off by a few roundings of 2^-24 of the
    running sum, which is at most that of the magnitudes; and what is added is rounded once more."""
    tol = 4e-7 * x.shape[1] ** 0.5 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -23 * (want.abs() + added.abs()) + 1e-6
    assert torch.equal(got.isnan(), want.isnan())
    assert ((got.double() - want).nan_to_num().abs() <= tol).all()


@pytest.mark.parametrize("depth", [8, 56, 64, 72, 768, 1024, 1032, 2048, 2056, 3072, 4000, 8192])
@pytest.mark.parametrize("rows,features", [(1, 8), (3, 12), (16, 1001), (8, 4100), (2, 260)])
def test_stored_rows(depth, rows, features):
    x, w = draw(1, rows, depth).bfloat16(), draw(2, features, depth, scale=0.05).bfloat16()
    bias, residual = draw(3, features), draw(4, rows, features)
    added = bias.double() + residual.double()
    close(K.gemm(x, w, bias=bias, residual=residual, out_f32=True, algo=3), x.double() @ w.double().T + added, x, w, added)


@pytest.mark.parametrize("depth,rows,features", [(768, 1, 2304), (768, 9, 3073), (2048, 16, 6144), (1000, 5, 520), (4096, 2, 264)])
def test_norm(depth, rows, features):
    x, w = draw(1, rows, depth), draw(2, features, depth, scale=0.05).bfloat16()
    gamma, beta = draw(3, depth), draw(4, depth)
    assert K.can_fuse_norm(rows, features, depth, torch.bfloat16)
    for g, b in ((gamma, beta), (gamma, None), (None, None)):
        h = torch.nn.functional.layer_norm(x.double(), (depth,), None if g is None else g.double(), None if b is None else b.double(), 1e-5)
        got = K.gemm(K.NormInput(x, g, b, 1e-5), w, out_f32=True)
        # rows rounded to bfloat16: 2^-9 of each number at most, at random: six times the deviation of their sum
        spread = 2.0 ** -9 * (h.square() @ w.double().square().T).sqrt()
        assert ((got.double() - h @ w.double().T).abs() <= 6 * spread + 1e-5).all()


@pytest.mark.parametrize("depth", [520, 768, 2048, 8192])
def test_rows_of_weights_stay_apart(depth):
    """An infinity and a NaN in a row of W reach its own feature alone, whatever the other halves of a tile hold."""
    x, w = draw(1, 4, depth).abs().bfloat16(), draw(2, 2048, depth, scale=0.05).bfloat16()
    w[9, depth - 8] = float("inf")
    w[2047, 0] = float("nan")
    got = K.gemm(x, w, out_f32=True, algo=3)
    assert got[:, 9].isinf().all() and got[:, 2047].isnan().all()
    got[:, 9] = 0
    got[:, 2047] = 0
    assert got.isfinite().all()


def test_operands_off_16_bytes():
    x, w = draw(1, 4, 768).bfloat16(), draw(2, 768, 768, scale=0.05).bfloat16()
    bias, residual = draw(3, 769)[1:], draw(4, 4 * 768 + 2)[2:].view(4, 768)
    added = bias.double() + residual.double()
    close(K.gemm(x, w, bias=bias, residual=residual, out_f32=True, algo=3), x.double() @ w.double().T + added, x, w, added)
