"""Shapes of the decode attention kernel, as the host chooses them for 256 compute units (also where no GPU is visible)."""
from types import SimpleNamespace

import pytest
import torch


@pytest.mark.parametrize("heads,rows", [(32, 8), (16, 16), (32, 1), (12, 20)])
@pytest.mark.parametrize("span,window", [(60, 0), (400, 0), (2048, 256)])
def test_rows_of_few_keys_are_one_workgroup_of_four_waves(monkeypatch, heads, rows, span, window):
    """More waves than a few keys give work to only make the merge of their results longer (60 keys: 5.6 us with four, 6.3 with eight)."""
    from swifttransformer_amd.parts import PartSpec, attention, build_part
    monkeypatch.setattr(attention, "_target_workgroups", lambda: 256)
    part = build_part("mixer", PartSpec("paged_attention", {"num_heads": heads, "head_dim": 64, "scale": 0.125, "bias": False, "window": window},
                                        {f"{n}.weight": n for n in ("q", "k", "v", "out")}), heads * 64, torch.bfloat16)
    assert part._shape_row_kernel(SimpleNamespace(max_kv_len=span), rows) == (1, 4)


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("heads,head_dim,dtype,rows,window,with_merge,without", [
    (12, 64, torch.bfloat16, 1, 0, 1, 1),        # 192 keys are 6 passes of a workgroup,
    (12, 80, torch.bfloat16, 1, 0, 3, 1),        # 12: three splits of four passes where the projection merges them
    (12, 128, torch.bfloat16, 4, 0, 3, 1),
    (12, 144, torch.bfloat16, 1, 0, 6, 1),       # 24
    (12, 256, torch.bfloat16, 8, 0, 3, 1),       # (three splits are what these rows have for all contexts)
    (12, 64, torch.float32, 1, 0, 3, 1),
    (12, 80, torch.float32, 1, 0, 6, 6),
    (12, 144, torch.float32, 1, 0, 8, 8),        # 48: eight splits, as for all contexts
    (12, 256, torch.float32, 1, 300, 1, 1),      # a window that is one split for all contexts
    (32, 256, torch.float32, 8, 0, 1, 1),        # a workgroup a unit
])
def test_splits_of_short_contexts(monkeypatch, heads, head_dim, dtype, rows, window, with_merge, without, fused):
    """A recorded step for up to 192 of 2,048 tokens."""
    from swifttransformer_amd.parts import PartSpec, attention, build_part
    from swifttransformer_amd.parts.base import KeySpan
    monkeypatch.setattr(attention, "_target_workgroups", lambda: 256)
    monkeypatch.setattr(attention.K, "can_fuse_merge", lambda *a: fused)
    part = build_part("mixer", PartSpec("paged_attention", {"num_heads": heads, "head_dim": head_dim, "scale": 0.125, "bias": False, "window": window},
                                        {f"{n}.weight": n for n in ("q", "k", "v", "out")}), heads * head_dim, dtype)
    assert part._shape_row_kernel(KeySpan(192, 2048), rows) == (with_merge if fused else without, 4)
    if rows * heads < 256 and not window:
        assert part._shape_row_kernel(KeySpan(192), rows)[0] == 1 and part._shape_row_kernel(KeySpan(2048, 2048), rows)[0] > 1


@pytest.mark.parametrize("rows,heads,window,same", [(8, 32, 0, True), (7, 32, 0, False), (1, 12, 0, False), (1, 12, 300, True), (16, 32, 0, True)])
def test_steps_of_one_shape(monkeypatch, rows, heads, window, same):
    """What decides whether short contexts have a recording of their own: the mixers' answers for both spans, whichever mixer it is."""
    from swifttransformer_amd.parts import PartSpec, attention, build_part
    from swifttransformer_amd.parts.base import CacheNeed, KeySpan, Mixer, decode_shape
    monkeypatch.setattr(attention, "_target_workgroups", lambda: 256)
    monkeypatch.setattr(attention.K, "can_fuse_merge", lambda *a: True)
    part = build_part("mixer", PartSpec("paged_attention", {"num_heads": heads, "head_dim": 64, "scale": 0.125, "bias": False, "window": window},
                                        {f"{n}.weight": n for n in ("q", "k", "v", "out")}), heads * 64, torch.bfloat16)
    differ = lambda m: decode_shape(m, KeySpan(192, 2048), rows) != decode_shape(m, KeySpan(2048, 2048), rows)
    assert differ(part) != same

    class Other(Mixer):
        def __init__(self, need):
            self.need = need

        def cache_need(self):
            return self.need
    assert not differ(Other(None)) and not differ(Other(CacheNeed("state", state_shape=(4,), state_dtype=torch.float32)))
    assert differ(Other(CacheNeed("paged_kv", num_kv_heads=1, head_dim=64))) and differ(object())
