"""Row kernels that take several columns and rows a thread, beside the same kernels on operands that no wide access fits: the same bits."""
import pytest
import torch

from test_zimorax_gpu import DEV, DTYPES, items_ctx

pytestmark = pytest.mark.gpu


def _shifted(t):
    """The same values, contiguous, four bytes (two in bfloat16) past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)[1:1 + t.numel()].view(t.shape)
    return flat.copy_(t)


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("in_dtype,out_dtype", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("width,lens", [(4, (70,)), (1028, (1, 2, 3, 61)), (8, (5, 1, 1, 1, 64, 2)), (2048, (63,)), (260, (1, 1, 1))])
def test_token_conv_in_pieces_of_four(taps, in_dtype, out_dtype, width, lens):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(width + taps)
    T = sum(lens) + 1                                          # and a padding row
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    wide = rnd(T, width + 5).to(in_dtype)
    x = torch.empty(T, width + 8, dtype=in_dtype, device=DEV)[:, 4:4 + width].copy_(wide[:, 1:1 + width])
    w, bias, state = rnd(width, taps), rnd(width), rnd(len(lens), taps - 1, width)
    ti, ln, off, sl = items_ctx(list(lens), list(range(len(lens)))[::-1])
    ti = torch.cat([ti, torch.full((1,), -1, dtype=torch.int32, device=DEV)])
    for kw in ({}, {"add_input": False, "bias": bias, "activation": "silu"}):
        s1, s2 = state.clone(), state.clone()
        four = K.token_conv(x, w, s1, (ti, ln, off, sl), out_dtype, **kw)
        one = K.token_conv(wide[:, 1:1 + width], w, s2, (ti, ln, off, sl), out_dtype, **kw)
        assert torch.equal(four, one) and torch.equal(s1, s2)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("rows,width", [(1, 4), (3, 1024), (70, 1028), (2, 2052)])
def test_dynamic_tanh_and_concat_cast_in_pieces_of_four(dtype, rows, width):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(width)
    dt = DTYPES[dtype]
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, base, w, b, w2, b2, alpha = rnd(rows, width), rnd(rows, width), rnd(width), rnd(width), rnd(width), rnd(width), rnd(1)
    picked = torch.randint(-1, rows, (rows + 2,), generator=g, device=DEV, dtype=torch.int32)

    def run(shift):
        f = _shifted if shift else (lambda t: t)
        outs = [torch.full((rows, width), 3.0, device=DEV), torch.full((rows, width), 3.0, device=DEV, dtype=dt),
                torch.full((rows + 2, width), 3.0, device=DEV, dtype=dt)]
        K.dynamic_tanh(f(x), w, b, alpha, out_f32=outs[0], out_t=outs[1], base=base, then=(w2, b2, alpha))
        K.dynamic_tanh(f(x), w, None, alpha, out_t=outs[2], rows=picked)
        return outs + [K.concat_cast(f(x), base, dt)]
    for four, one in zip(run(False), run(True)):
        assert torch.equal(four, one)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("heads,hd,splits,gated", [(12, 64, 16, False), (3, 16, 2, True), (2, 80, 9, True), (1, 256, 70, False), (4, 128, 64, True)])
def test_split_attention_merged_by_lanes(dtype, heads, hd, splits, gated):
    """Rows whose keys are shared out over many splits, some of them empty (3 to 90 keys on up to 70 splits), against one split."""
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(splits)
    dt, ps, lens = DTYPES[dtype], 16, (3, 90, 17)
    B = len(lens)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    kc, vc = rnd(8 * B, heads, ps, hd).to(dt), rnd(8 * B, heads, ps, hd).to(dt)
    bt = torch.arange(8 * B, device=DEV, dtype=torch.int32).view(B, 8)
    q, item = rnd(B, heads * hd).to(dt), torch.arange(B, device=DEV, dtype=torch.int32)
    pos = torch.tensor(lens, device=DEV, dtype=torch.int32) - 1
    kw = {"head_gate": rnd(B, heads)} if gated else {}
    one = K.attention_rows(q, kc, vc, item, pos, bt, heads, hd ** -0.5, num_splits=1, **kw)
    many = K.attention_rows(q, kc, vc, item, pos, bt, heads, hd ** -0.5, num_splits=splits, **kw)
    # float sums of up to 90 weights in another order, then one rounding to the storage type (2^-9 of a value up to twice)
    tol = 1e-5 if dt == torch.float32 else 2.0 ** -8
    assert bool(((one.float() - many.float()).abs() <= tol * one.float().abs() + 1e-5).all())


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("splits", [1, 4, 64, 70])
def test_a_value_that_is_no_number_reaches_the_result_of_every_split(dtype, splits):
    """A visible key whose weight is down to zero beside another split's, with a NaN or an infinity in its value (zero times either is NaN):
    the result shows it however many splits the keys are shared out over, and splits without a key show nothing."""
    from swifttransformer_amd.ops import kernels as K
    dt, ps, hd, n = DTYPES[dtype], 16, 64, 80
    q = torch.zeros(1, hd, device=DEV, dtype=dt)
    q[0, 0] = 1.0
    kc, vc = torch.zeros(6, 1, ps, hd, device=DEV, dtype=dt), torch.ones(6, 1, ps, hd, device=DEV, dtype=dt)
    kc[4, 0, 15, 0] = 4000.0                                   # the last key has all of the weight
    vc[0, 0, 3, 5], vc[1, 0, 7, 9] = float("nan"), float("inf")
    kc[5], vc[5] = float("nan"), float("nan")                  # nobody's page
    bt = torch.arange(6, device=DEV, dtype=torch.int32).view(1, 6)
    item, pos = torch.zeros(1, dtype=torch.int32, device=DEV), torch.full((1,), n - 1, dtype=torch.int32, device=DEV)
    out = K.attention_rows(q, kc, vc, item, pos, bt, 1, 1.0, num_splits=splits)[0]
    bad = torch.isnan(out).nonzero().flatten().tolist()
    assert bad == [5, 9] and bool((out[~torch.isnan(out)] == 1.0).all())


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("heads,kv_heads,hd", [(1, 1, 16), (32, 8, 64), (33, 3, 64), (12, 12, 80), (32, 32, 128), (16, 17, 64)])
def test_normed_queries_and_keys_in_pieces(dtype, heads, kv_heads, hd):
    """Rows in registers (up to 4,096 numbers) beside the same rows past a 16-byte boundary, which go a number at a time, with padding rows."""
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(heads + hd)
    dt, ps, T = DTYPES[dtype], 16, 5
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    qk, gq, gk = rnd(T, (heads + kv_heads) * hd), rnd(heads * hd), rnd(kv_heads * hd)
    item = torch.tensor([0, 1, -1, 0, 1], dtype=torch.int32, device=DEV)
    pos = torch.tensor([0, 17, 3, 1, -1], dtype=torch.int32, device=DEV)
    bt = torch.tensor([[2, 0], [1, 3]], dtype=torch.int32, device=DEV)
    res = []
    for shift in (False, True):
        k, v = torch.full((4, kv_heads, ps, hd), 7.0, dtype=dt, device=DEV), torch.full((4, kv_heads, ps, hd), 7.0, dtype=dt, device=DEV)
        f = _shifted if shift else (lambda t: t)
        q = K.qk_norm_write(qk, f(gq), f(gk), 1e-5, heads, kv_heads, hd, k, v, item, pos, bt, write=True)
        res.append((q.clone(), k, v))
    # two float sums of up to 4,096 squares in different orders, then one rounding (to either side of a half at most)
    tol = 2e-6 if dt == torch.float32 else 2.0 ** -7
    for a, b in zip(*res):
        assert bool(((a.float() - b.float()).abs() <= tol * b.float().abs()).all())
    assert torch.equal(res[0][2], res[1][2])


@pytest.mark.parametrize("streams", [1, 4, 5, 6, 8])        # (six and eight with 256 threads whatever the rows)
@pytest.mark.parametrize("rows,width", [(1, 4), (3, 1028), (2, 2048), (2, 8196), (300, 516)])
def test_streams_written_by_as_many_threads_as_columns(streams, rows, width):
    from swifttransformer_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(width + streams)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, y, mix, b, a2, gain = rnd(rows, streams, width), rnd(rows, width), rnd(streams, streams), rnd(streams), rnd(streams), rnd(width)
    new = torch.einsum("rsw,st->rtw", x.double(), mix.double()) + b.double()[None, :, None] * y.double()[:, None]
    size = torch.einsum("rsw,st->rtw", x.double().abs(), mix.double().abs()) + (b.double()[None, :, None] * y.double()[:, None]).abs()
    u, u_size = torch.einsum("rtw,t->rw", new, a2.double()), torch.einsum("rtw,t->rw", size, a2.double().abs())
    norm = torch.sqrt(u.square().mean(1, keepdim=True) + 1e-5)
    got = x.clone().view(rows, streams * width)
    out = K.streams_write(got, y, mix, b, then=(a2, gain, 1e-5), out_dtype=torch.float32)
    # chains of a few float operations a number; the norm's sum of squares adds its own few roundings, relative
    assert bool(((got.view_as(x).double() - new).abs() <= 1e-6 * size + 1e-30).all())
    assert bool(((out.double() - u / norm * gain.double()).abs() <= (2e-6 * u_size + 2e-5 * u.abs()) / norm * gain.double().abs() + 1e-30).all())


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("in_dtype,out_dtype", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("width,lens", [(1028, (1, 2, 3, 1, 514)), (516, (1029,)), (2052, (200, 1, 1, 1, 139, 3))])
def test_token_conv_with_four_rows_a_thread(taps, in_dtype, out_dtype, width, lens):
    """Rows enough for every compute unit, items that begin anywhere in a thread's four rows, a last group that is not whole, a padding row."""
    from swifttransformer_amd.ops import kernels as K
    T = sum(lens) + 1
    assert -(-T // 4) * -(-width // 1024) >= torch.cuda.get_device_properties(0).multi_processor_count
    g = torch.Generator(device=DEV).manual_seed(width + taps)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    wide = rnd(T, width + 5).to(in_dtype)
    x = torch.empty(T, width + 8, dtype=in_dtype, device=DEV)[:, 4:4 + width].copy_(wide[:, 1:1 + width])
    w, bias, state = rnd(width, taps), rnd(width), rnd(len(lens), taps - 1, width)
    ti, ln, off, sl = items_ctx(list(lens), list(range(len(lens)))[::-1])
    ti = torch.cat([ti, torch.full((1,), -1, dtype=torch.int32, device=DEV)])
    for kw in ({}, {"add_input": False, "bias": bias, "activation": "silu"}):
        s1, s2 = state.clone(), state.clone()
        four = K.token_conv(x, w, s1, (ti, ln, off, sl), out_dtype, **kw)
        one = K.token_conv(wide[:, 1:1 + width], w, s2, (ti, ln, off, sl), out_dtype, **kw)
        assert torch.equal(four, one) and torch.equal(s1, s2)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("rows,width", [(130, 2052), (300, 516), (257, 4)])
def test_dynamic_tanh_of_many_rows_in_pieces_of_four(dtype, rows, width):
    from swifttransformer_amd.ops import kernels as K
    assert rows * -(-width // 1024) > torch.cuda.get_device_properties(0).multi_processor_count
    g = torch.Generator(device=DEV).manual_seed(width)
    dt = DTYPES[dtype]
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, base, w, b, w2, b2, alpha = rnd(rows, width), rnd(rows, width), rnd(width), rnd(width), rnd(width), rnd(width), rnd(1)
    picked = torch.randint(-1, rows, (rows + 2,), generator=g, device=DEV, dtype=torch.int32)

    def run(shift):
        f = _shifted if shift else (lambda t: t)
        outs = [torch.full((rows, width), 3.0, device=DEV), torch.full((rows, width), 3.0, device=DEV, dtype=dt),
                torch.full((rows + 2, width), 3.0, device=DEV, dtype=dt)]
        K.dynamic_tanh(f(x), w, b, alpha, out_f32=outs[0], out_t=outs[1], base=base, then=(w2, b2, alpha))
        K.dynamic_tanh(f(x), w, None, alpha, out_t=outs[2], rows=picked)
        return outs
    for four, one in zip(run(False), run(True)):
        assert torch.equal(four, one)
