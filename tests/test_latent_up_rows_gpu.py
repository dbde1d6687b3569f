"""Decoded tokens' read-out of a latent: key splits merged, a head's product and its gate, in registers and past what they hold; against float64."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# values, entries, splits: up to 128, 128 and 64 are one kernel's, the rest the other's
@pytest.mark.parametrize("vd,od,splits", [(1, 16, 1), (33, 112, 8), (96, 80, 9), (128, 128, 16), (128, 128, 64), (128, 128, 65), (129, 128, 3), (64, 144, 5), (64, 48, 40), (80, 64, 17)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_splits_product_and_gate(vd, od, splits, dtype):
    g = torch.Generator().manual_seed(vd * 100 + od + splits)
    T, H = 5, 3
    part, lse = torch.randn(T, H, splits, od, generator=g), torch.randn(T, H, splits, generator=g) * 3
    lse[1, 0, 0] = float("-inf")                     # a split without a key (one split: a row without any)
    lse[2, 1] = float("-inf")
    w = (torch.randn(H, vd, od, generator=g) * od ** -0.5).to(dtype)
    wide = torch.randn(T, H * vd + 3, generator=g)
    item = torch.tensor([0, 1, 2, -1, 3], dtype=torch.int32, device=DEV)
    weight = torch.nan_to_num(torch.softmax(lse.double(), dim=2), nan=0.0)
    o = (weight[..., None] * part.double()).sum(2)
    up = torch.einsum("thr,hvr->thv", o, w.double())
    po, pl, wd, zd = part.to(DEV), lse.to(DEV), w.to(DEV), wide.to(DEV)
    # float sums of the splits and of the entries; half of 2^-8 of a bfloat16 result
    bound = 4e-7 * (splits ** 0.5 + od ** 0.5) * torch.einsum("thr,hvr->thv", (weight[..., None] * part.double().abs()).sum(2), w.double().abs()) + 1e-7
    for gate in (False, True):
        want = up * torch.sigmoid(wide[:, 1:1 + H * vd].double().view(T, H, vd)) if gate else up
        y = torch.full((T, H * vd), 7.0, dtype=dtype, device=DEV)
        K._check(K._lib().st_latent_up(K._ptr(y), None, K._ptr(po), K._ptr(pl), splits, K._ptr(wd), K._ptr(zd[:, 1:]) if gate else None, zd.stride(0), K._ptr(item),
                                       T, H, vd, od, K.dtype_code(dtype), K._stream()))
        got = y.cpu().double().view(T, H, vd)
        assert (got[3] == 7.0).all()
        tol = bound + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)
        rows = [0, 1, 2, 4]
        assert ((got - want).abs() <= tol)[rows].all()
