"""bfloat16 products whose depth is dealt to several workgroups: rows and features at the edges of their tiles, depths that their parts do
not divide evenly, every epilogue; against float64.  And which products go there."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def draw(seed, *shape, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(DEV)


def bound(x, w, depth):
    """Exact products, summed in float in some order: a few roundings of 2^-24 of the running sum."""
    return 4e-7 * depth ** 0.5 * (x.double().abs() @ w.double().abs().T) + 1e-6


@pytest.mark.parametrize("rows,features,depth", [(1, 4, 128), (13, 128, 192), (63, 132, 256), (64, 260, 704), (65, 128, 1024), (96, 512, 2048), (129, 124, 640),
                                                 (160, 384, 1088), (193, 256, 512), (225, 200, 2048), (256, 2048, 256), (257, 128, 4096), (300, 516, 1024),
                                                 (449, 128, 8192), (512, 256, 128), (1000, 132, 320)])
def test_against_float64(rows, features, depth):
    x, w = draw(1, rows, depth).bfloat16(), draw(2, features, depth, scale=0.05).bfloat16()
    bias, residual = draw(3, features), draw(4, rows, features)
    base, tol = x.double() @ w.double().T, bound(x, w, depth)
    got = K.gemm(x, w, bias=bias, residual=residual, out_f32=True, algo=4)
    assert ((got.double() - (base + bias.double() + residual.double())).abs() <= tol).all()
    got = K.gemm(x, w, bias=bias, residual=residual, out_f32=True, algo=4, out_scale=0.25, bias_unscaled=True)
    assert ((got.double() - (0.25 * base + bias.double() + residual.double())).abs() <= tol).all()
    for act, f in (("relu", torch.relu), ("gelu", lambda v: torch.nn.functional.gelu(v)), ("relu_squared", lambda v: torch.relu(v).square())):
        want = f(base + bias.double())
        got = K.gemm(x, w, bias=bias, activation=act, algo=4).double()
        # bfloat16 results: half of 2^-8 of each; the functions' slope is at most twice their argument
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + tol * 2 * (1 + (base + bias.double()).abs())).all(), act


def test_rows_and_features_stay_apart():
    """NaN in a row of x reaches that row's results alone, an infinity in a row of W that feature's, also where a tile ends past them."""
    x, w = draw(1, 70, 1024).abs().bfloat16(), draw(2, 132, 1024, scale=0.05).bfloat16()
    x[69, 3] = float("nan")
    w[131, 1000] = float("inf")
    got = K.gemm(x, w, out_f32=True, algo=4)
    assert got[69].isnan().all() and got[:69, 131].isinf().all() and got[:69, :131].isfinite().all()


@pytest.mark.parametrize("rows,features,depth,taken", [(64, 2048, 8192, False), (65, 2048, 8192, True), (512, 2048, 8192, True), (513, 2048, 8192, True), (577, 2048, 16384, True), (768, 768, 8192, True),
                                                       (769, 768, 8192, False), (576, 1024, 4096, False), (577, 4096, 8192, False), (150, 4096, 16384, True), (12, 4096, 16384, False),
                                                       (64, 2048, 2048, False), (150, 8192, 2048, False), (100, 2560, 10240, True), (100, 2560, 10208, False)])
def test_which_products_go_there(rows, features, depth, taken):
    x, w = draw(1, rows, depth).bfloat16(), draw(2, features, depth, scale=0.05).bfloat16()
    residual = draw(4, rows, features)
    K.gemm_parts_count(reset=True)
    got = K.gemm(x, w, residual=residual, out_f32=True)
    assert K.gemm_parts_count() == int(taken)
    assert ((got.double() - (x.double() @ w.double().T + residual.double())).abs() <= bound(x, w, depth)).all()
    if taken:                                        # operands off 16 bytes go where they went
        wide = torch.empty(rows * depth + 1, dtype=torch.bfloat16, device=DEV)
        off = wide[1:].view(rows, depth).copy_(x)
        assert torch.allclose(K.gemm(off, w, residual=residual, out_f32=True), got, rtol=1e-4, atol=1e-3)
        assert K.gemm_parts_count() == 1
