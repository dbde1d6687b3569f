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
