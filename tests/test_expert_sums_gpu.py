"""Routed experts of one and two tokens, whose output product sums over a token's choices itself: the same numbers, to the last bit, as the
same tokens get among more of them (output product, pairs' results, sum)."""
import pytest
import torch

from swifttransformer_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,F,E,top,style,identity,clamped", [
    (64, 64, 16, 2, "softmax_output", 0, False),
    (72, 40, 6, 1, "sigmoid_output", 0, False),          # part of a block of features; one choice
    (20, 28, 5, 3, "softmax_corrected", 2, True),        # depths of no whole pieces; identity experts
    (1000, 520, 8, 4, "softmax_all", 0, False),
    (96, 2056, 7, 2, "scaled_input", 0, False),          # weights on the inputs
    (96, 520, 7, 2, "scaled_input", 0, False),           # (the rows before are too long for the kernel)
    (64, 64, 9, 5, "softmax_output", 0, False),          # more choices than the kernel takes
])
def test_few_tokens(dtype, W, F, E, top, style, identity, clamped):
    g = torch.Generator(device="cuda").manual_seed(W + F + E)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std)
    x, wu, wd = rnd(4, W).to(dtype), rnd(E, F, W, std=W ** -0.5).to(dtype), rnd(E, W, F, std=F ** -0.5).to(dtype)
    wg = None if style == "sigmoid_output" else rnd(E, F, W, std=W ** -0.5).to(dtype)
    logits, corr = rnd(4, E + identity), rnd(E + identity)
    if identity:
        logits[0, E:] += 9.0                             # a token of identity experts (and one more choice)
    residual = rnd(4, W)
    for item in (torch.zeros(4, dtype=torch.int32, device="cuda"), torch.tensor([-1, 0, 0, 0], dtype=torch.int32, device="cuda")):
        def run(n, res):
            return K.routed_experts(x[:n], logits[:n], wg, wu, wd, res, top=top, limit=0.9, out_scale=0.75, token_item=item[:n], style=style,
                                    groups=4 if style == "softmax_all" else 1, keep=2 if style == "softmax_all" else 1, correction=corr, scale=1.5,
                                    identity=identity, clamped=clamped)
        many = run(4, residual.clone())
        for n in (1, 2):
            assert torch.equal(run(n, residual[:n].clone()), many[:n])
        if style != "scaled_input":
            many = run(4, None)
            for n in (1, 2):
                assert torch.equal(run(n, None), many[:n])
    assert bool(torch.isfinite(many).all()) and float(many.abs().max()) > 0


@pytest.mark.parametrize("dtype,W,F,top,one,two", [
    (torch.bfloat16, 768, 768, 4, True, True), (torch.float32, 768, 768, 3, False, True),
    (torch.bfloat16, 1024, 4096, 1, True, True), (torch.bfloat16, 1024, 4096, 2, False, False),      # few workgroups, long rows
    (torch.float32, 2048, 2048, 1, True, True), (torch.float32, 2048, 2056, 1, True, False),         # 16 MB and more a matrix
    (torch.bfloat16, 2048, 2048, 3, True, True), (torch.bfloat16, 2048, 2048, 4, False, True),
    (torch.bfloat16, 64, 64, 5, False, False),
])
def test_which_sizes_are_summed_so(dtype, W, F, top, one, two):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the line depends on the number of compute units")
    assert [bool(K._lib().st_moe_down_sum_offered(n, top, W, F, K.dtype_code(dtype))) for n in (1, 2, 3)] == [one, two, False]
