"""Float products on the bfloat16 matrix cores (csrc/gemm_f32.hip) against float64.

Bound of an element's error: every 16 in depth take a rounding of the sum of the largest parts' products, and what is left of the depth one
a number; a rounding is at most 2^-24 of a sum that never exceeds S = sum |x| |w|; the other products' sum is at most 2^-7 of S, with five
times as many roundings; the products left out are at most 2^-25 of S; the merge of chains and splits, bias, residual and factor add a dozen
more."""
import pytest
import torch

from swifttransformer_amd.ops import arena
from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


def operands(M, N, D, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + M * 7 + N * 3 + D)
    x = torch.empty(M, D, device="cuda").normal_(0, 1, generator=g)
    w = torch.empty(N, D, device="cuda").normal_(0, 0.05, generator=g)
    return x, w, g


def parted(M, N, D):
    """Whether the product has tiles that are parted over the depth and summed (it asks for room for their sums)."""
    return K._gemm_scratch(M, N, D, 0, False, 3) > 0


def check(y, x, w, bias=None, residual=None, scale=1.0, extra=0.0):
    ref = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    if bias is not None:
        ref, size = ref + bias.double(), size + bias.double().abs()
    ref, size = ref * scale, size * abs(scale)
    if residual is not None:
        ref, size = ref + residual.double(), size + residual.double().abs()
    D = x.shape[1]
    roundings = D // 16 * (1 + 5 * 2.0 ** -7) + D % 32 + 12
    bound = (roundings * 2.0 ** -24 + 2.0 ** -25) * size
    over = ((y.double() - ref).abs() > bound + extra)
    assert not bool(over.any()), float(((y.double() - ref).abs() / bound).max())


# edges of the 128 x 128 tiles, depths that are no whole steps of 32, tiles in whole rounds, split ones and both (256 compute units)
@pytest.mark.parametrize("M,N,D,parts", [
    (1, 4, 4, False), (3, 12, 28, False), (127, 132, 32, False), (128, 128, 36, False), (129, 124, 64, False), (200, 260, 100, False), (96, 512, 96, False),
    (257, 1028, 516, True), (701, 5376, 512, False), (701, 6144, 512, True), (1000, 4100, 1000, True), (130, 2048, 4096, True), (1, 4, 2052, True)])
def test_shapes(M, N, D, parts):
    assert parted(M, N, D) == parts
    x, w, g = operands(M, N, D)
    bias = torch.empty(N, device="cuda").normal_(0, 1, generator=g)
    check(K.gemm(x, w, algo=3), x, w)
    check(K.gemm(x, w, bias=bias, algo=3), x, w, bias=bias)


def test_chosen_and_closer_than_the_library():
    """The rule sends a prompt's product here; it is closer to float64 than the library's float product."""
    x, w, _ = operands(701, 2048, 2048)
    assert K._gemm_scratch(701, 2048, 2048, 0, False) > 0 and K._gemm_scratch(64, 2048, 2048, 0, False) == 0
    ref = x.double() @ w.double().T
    K.gemm_path_counts(reset=True), K.gemm_split_count(reset=True)
    own, lib = K.gemm(x, w), K.gemm(x, w, algo=2)
    assert K.gemm_split_count() == 1 and {n: c for n, c in K.gemm_path_counts().items() if c} == {"library": 1}
    assert torch.equal(own, K.gemm(x, w, algo=3)) and torch.equal(own, K.gemm(x, w))
    assert float((own - ref).norm()) < float((lib - ref).norm())


@pytest.mark.parametrize("M,N,D", [(300, 512, 256), (701, 2048, 2048), (200, 2048, 8192)])
@pytest.mark.parametrize("share", [1.0, 0.5, 0.1, 0.02, 0.005])
def test_no_further_off_than_the_library(M, N, D, share):
    """Also where most of x is zero (activations behind a ReLU): a product takes no more roundings of the running sum than a float product."""
    x, w, g = operands(M, N, D)
    x = torch.where(torch.rand(M, D, device="cuda", generator=g) < share, x, 0.0)
    ref = x.double() @ w.double().T
    own, lib = ((K.gemm(x, w, algo=a).double() - ref).norm() for a in (3, 2))
    assert float(own) < float(lib)


@pytest.mark.parametrize("M,N,D,taken", [
    (96, 2560, 10240, False), (97, 2560, 10240, True), (128, 8192, 2048, False), (140, 10240, 2560, False), (200, 2048, 8192, True), (256, 4096, 4096, True),
    (300, 6144, 2048, False), (300, 2048, 8192, True), (300, 4096, 4096, False), (701, 6144, 2048, True), (2048, 3072, 768, False), (2048, 2048, 2048, True)])
def test_which_sizes_are_taken(M, N, D, taken):
    """Those that are no slower than in the library (the figures are beside the rule)."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the line depends on the number of compute units")
    x, w, _ = operands(M, N, D)
    K.gemm_path_counts(reset=True), K.gemm_split_count(reset=True)
    K.gemm(x, w)
    assert (K.gemm_split_count(), K.gemm_path_counts()["library"]) == (int(taken), int(not taken))


def test_most_scratch_of_smaller_steps():
    assert K._gemm_scratch(1024, 2048, 2048, 0, True) >= max(K._gemm_scratch(m, 2048, 2048, 0, False) for m in range(1, 1025))
    assert not arena.measuring()


# (every epilogue of the kernel and of the sum of parted tiles)
@pytest.mark.parametrize("M,N,D,parts", [(300, 256, 516, True), (701, 2048, 512, False), (701, 2048, 2048, True)])
def test_epilogues(M, N, D, parts):
    assert parted(M, N, D) == parts
    x, w, g = operands(M, N, D)
    bias = torch.empty(N, device="cuda").normal_(0, 1, generator=g)
    residual = torch.empty(M, N, device="cuda").normal_(0, 1, generator=g)
    plain = K.gemm(x, w, algo=3)
    check(K.gemm(x, w, bias=bias, residual=residual, out_scale=0.5, algo=3), x, w, bias, residual, 0.5)
    check(K.gemm(x, w, residual=residual, algo=3), x, w, residual=residual)
    assert torch.equal(K.gemm(x, w, activation="relu", algo=3), plain.clamp(min=0))
    y = K.gemm(x, w, bias=bias, activation="gelu", algo=3)
    z = x.double() @ w.double().T + bias.double()
    want = 0.5 * z * (1 + torch.erf(z / 2 ** 0.5))
    assert float((y - want).abs().max()) <= 1e-5 * float(z.abs().max())
    unscaled = K.gemm(x, w, bias=bias, out_scale=0.5, bias_unscaled=True, algo=3)
    check(unscaled, x, w * 0.5, bias=bias)


@pytest.mark.parametrize("M,D,parts", [(130, 256, False), (701, 256, False), (701, 1024, True)])
def test_pages(M, D, parts):
    """A fused query, key and value product writes its pages as the library's product and the page write do."""
    heads, hd, page = 4, 32, 8
    N = 3 * heads * hd
    assert parted(M, N, D) == parts
    x, w, _ = operands(M, N, D)
    pages = -(-M // page) + 2
    table = torch.randperm(pages, device="cuda").int()[None].contiguous()
    item = torch.zeros(M, dtype=torch.int32, device="cuda")
    item[5] = -1                                                    # a padding row
    pos = torch.arange(M, dtype=torch.int32, device="cuda")
    made = []
    for algo in (2, 3):
        kc, vc = (torch.zeros(pages, heads, page, hd, device="cuda") for _ in range(2))
        y = K.gemm(x, w, algo=algo, kv_scatter=K.KvScatter(kc, vc, item, pos, table, heads * hd))
        made.append((y, kc, vc))
    check(made[1][0], x, w)
    at = (table[0].long()[pos.long() // page], pos.long() % page)
    rows = torch.arange(M, device="cuda") != 5
    for c, part in ((made[1][1], made[1][0][:, heads * hd:2 * heads * hd]), (made[1][2], made[1][0][:, 2 * heads * hd:])):
        assert torch.equal(c[at[0], :, at[1]].reshape(M, -1)[rows], part[rows])
        assert bool((c[at[0][5], :, at[1][5]] == 0).all())
    assert torch.equal(made[0][1] != 0, made[1][1] != 0)


@pytest.mark.parametrize("D,parts", [(200, False), (1032, True)])
def test_numbers_that_parts_do_not_hold(D, parts):
    """Infinities, NaN, numbers past bfloat16's largest and tiny ones give what float products give, and other rows are as without."""
    M, N = 300, 256
    assert parted(M, N, D) == parts
    x, w, _ = operands(M, N, D)
    clean = K.gemm(x, w, algo=3)
    inf, big = float("inf"), 3.4e38
    x[3, 7], x[70, 0], x[140, 199], x[200, 5] = inf, -inf, float("nan"), big
    w[9, 5] = 0.0
    x[250] *= 2.0 ** -120
    y = K.gemm(x, w, algo=3)
    ref = x.double() @ w.double().T
    for r in (3, 70):
        assert torch.equal(y[r], ref[r].float())
    assert bool(torch.isnan(y[140]).all())
    held = ref[200].abs() < 3e38
    size = x[200].double().abs() @ w.double().abs().T
    assert bool(((y[200].double() - ref[200]).abs()[held] <= 2.0 ** -20 * size[held]).all())
    size = x[250].double().abs() @ w.double().abs().T
    assert bool(((y[250].double() - ref[250]).abs() <= (D + 12) * 2.0 ** -24 * size + D * 2.0 ** -149).all())
    rows = torch.ones(M, dtype=torch.bool, device="cuda")
    rows[[3, 70, 140, 200, 250]] = False
    keep = torch.ones(N, dtype=torch.bool, device="cuda")
    keep[9] = False
    check(y[rows], x[rows], w)
    assert bool(torch.isfinite(clean).all())


# (splits: 701 rows of 2,048 x 2,048 are 96 tiles, parted over the depth; 300 of 256 x 200 are whole)
@pytest.mark.parametrize("M,N,D", [(300, 256, 200), (701, 2048, 2048)])
@pytest.mark.parametrize("tiny,large", [(-120, 40), (-130, 60), (-140, 60), (-136, 0), (-110, 100)])
def test_tiny_numbers_with_large_ones(M, N, D, tiny, large):
    """Numbers that three bfloat16 numbers do not hold, in rows of x and of W, times numbers that make ordinary sums of them: no further off
    than D roundings of a float sum."""
    assert parted(M, N, D) == (D > 1000)
    x, w, g = operands(M, N, D)
    normal = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g).double()
    x[5], x[M - 2] = (normal(D) * 2.0 ** tiny).float(), torch.where(torch.arange(D, device="cuda") == D - 40, 2.0 ** tiny * 1.2345678, 0.0)
    w[7], w[130] = (normal(D) * 2.0 ** large).float(), 2.0 ** large
    w[3], x[131] = (normal(D) * 2.0 ** tiny).float(), 2.0 ** large
    # some rows, all of x and all of W (sums that look ordinary everywhere)
    for a, b in ((x, w), ((normal(M, D) * 2.0 ** tiny).float(), (normal(N, D) * 2.0 ** large).float()),
                 ((normal(M, D) * 2.0 ** large).float(), (normal(N, D) * 2.0 ** tiny).float())):
        y = K.gemm(a, b, algo=3)
        ref, size = a.double() @ b.double().T, a.double().abs() @ b.double().abs().T
        over = (y.double() - ref).abs() > (D + 12) * 2.0 ** -24 * size + D * 2.0 ** -149
        held = ref.abs() < 2.0 ** 128                               # (large ones among themselves may be past float's range)
        assert not bool((over & held).any()), (over & held).nonzero()[:4].tolist()
        assert not bool(torch.isfinite(y[~held]).any())


@pytest.mark.parametrize("M,N,D", [(300, 256, 200), (701, 2048, 2048)])
def test_rows_do_not_change_each_other(M, N, D):
    """Infinities, NaN, numbers past bfloat16's largest and tiny ones in some rows of x: the others' results stay the same to the last bit."""
    assert parted(M, N, D) == (D > 1000)
    x, w, _ = operands(M, N, D)
    clean = K.gemm(x, w, algo=3)
    x[3, 7], x[70, 0], x[140, D - 1], x[200, 5], x[201, 3] = float("inf"), -float("inf"), float("nan"), 3.4e38, 1e-42
    x[250] *= 2.0 ** -120
    rows = torch.ones(M, dtype=torch.bool, device="cuda")
    rows[[3, 70, 140, 200, 201, 250]] = False
    y = K.gemm(x, w, algo=3)
    assert torch.equal(y[rows], clean[rows])
    assert not torch.equal(y[201], clean[201])


def test_without_room_for_the_sums():
    """A caller of the C entry that brings no scratch: the library, as before there was a kernel that asks for it; too little: the same."""
    import ctypes
    M, N, D = 200, 2048, 8192
    x, w, _ = operands(M, N, D)
    assert K._gemm_scratch(M, N, D, 0, False) > 4
    room, out = torch.empty(4, device="cuda"), torch.empty(M, N, device="cuda")
    ex = K._GemmExtras()
    ex.scratch, ex.scratch_floats = room.data_ptr(), 4
    for extras in (None, ctypes.byref(ex)):
        K.gemm_path_counts(reset=True), K.gemm_split_count(reset=True)
        assert K._lib().st_gemm(out.data_ptr(), x.data_ptr(), w.data_ptr(), None, None, M, N, D, 0, 0, 1, 0, extras,
                                torch.cuda.current_stream().cuda_stream) == 0
        assert K.gemm_path_counts()["library"] == 1 and K.gemm_split_count() == 0
        ref, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        assert bool(((out.double() - ref).abs() <= D * 2.0 ** -24 * size).all())


def test_rows_off_16_bytes_go_to_the_library():
    buf, _, _ = operands(1, 1, 701 * 2048 + 1)
    w = operands(4, 2048, 2048)[1]
    x = buf[0, 1:].view(701, 2048)
    assert x.data_ptr() % 16 == 4
    before = K.gemm_path_counts()["library"]
    check(K.gemm(x, w), x, w)
    assert K.gemm_path_counts()["library"] == before + 1
