"""Best tokens out of the head's own kernel behind norms that it does not know: the branch of the model's head step, and where it is not taken."""
import pytest
import torch

import tiny_gisedra as tiny
from test_zimorax_gpu import make_runner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_recorded_steps_find_their_best_tokens_behind_a_dynamic_tanh(tmp_path, monkeypatch, dtype):
    """A vocabulary wide enough for the kernel that walks over it (four tiles of 16 for every compute unit)."""
    from swifttransformer_amd.engine.step import StepEntry
    from swifttransformer_amd.ops import kernels as K
    units = torch.cuda.get_device_properties(0).multi_processor_count
    vocab = 64 * units + 13
    cfg = {"architecture": "Gisedra", "vocab": vocab, "width": 64, "max_positions": 512, "norm": {"eps": 1e-6},
           "layers": [tiny._with(tiny._latent(2, 24, 8, 16, 20, 0.3), None)]}
    asked, sampled = [], []
    gemm, sample = K.gemm, K.sample
    monkeypatch.setattr(K, "gemm", lambda *a, **k: (asked.append(k["best"].shape[0]) if k.get("best") is not None else None, gemm(*a, **k))[1])
    monkeypatch.setattr(K, "sample", lambda *a, **k: (sampled.append(1), sample(*a, **k))[1])
    runner = make_runner(tiny.write_folder(cfg, str(tmp_path / "m"), 3), dtype, 16, 12, max_seqs=3)
    head, norm = runner.model.head, runner.model.final_norm
    wide = dtype == "bfloat16"
    assert not head.takes_norm(3, norm) and head.offers_best(3) is wide and not head.offers_best(17)
    for r in range(3):
        runner.admit(r)
        runner.step([StepEntry(r, tiny.prompt(9 + 7 * r, vocab, r), [])])
    asked.clear(), sampled.clear()
    tokens = [5, 70, 900]
    for _ in range(4):                                # recorded, then replayed
        logits = runner.step([StepEntry(r, [tokens[r]], [0]) for r in range(3)])
        best = runner._recorded[3].best[:3].cpu()
        assert torch.equal(best.long(), logits.argmax(1).cpu())
        tokens = best.tolist()
    assert asked == ([3, 3] if wide else []) and len(sampled) == (0 if wide else 2)      # (once beforehand, once recorded)


@pytest.mark.parametrize("extra", [{"logit_scale": 0.5}, {"logit_scale": 2.0}, {"softcap": 30.0}, {"embed_dim": 72}])
def test_a_factor_a_limit_or_a_projection_behind_the_head_keeps_the_arg_max_kernel(extra):
    """They may make two different logits equal (or are a product of their own): the best is then found behind them."""
    from swifttransformer_amd.parts import PartSpec, build_part
    vocab = 64 * torch.cuda.get_device_properties(0).multi_processor_count + 13
    spec = {"vocab_size": vocab, "embed_dim": 64, "tied_to": None}
    build = lambda p: build_part("head", PartSpec("linear", p, {"weight": "w", "project_out": "p"}), 64, torch.bfloat16)
    assert build(spec).offers_best(1) and not build(dict(spec, **extra)).offers_best(1)
