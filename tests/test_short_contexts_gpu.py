"""Recorded decode steps of short contexts beside those of all: the step that a batch is given, and the results where a request
grows out of the short ones."""
import numpy as np
import pytest
import torch

import plain_opt
import tiny
from test_engine_gpu import DTYPES, check, make_runner

pytestmark = pytest.mark.gpu

CFG = dict(vocab_size=777, max_position_embeddings=1024, hidden_size=192, num_hidden_layers=2, num_attention_heads=3, ffn_dim=200,
           word_embed_proj_dim=192, do_layer_norm_before=True, enable_bias=True, tie_word_embeddings=True)


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    from swifttransformer_amd.config import OptHyperParam
    from swifttransformer_amd.weights import write_random_model
    d = write_random_model(OptHyperParam(**CFG).validate(), str(tmp_path_factory.mktemp("short") / "m"), seed=3)
    return (d,) + plain_opt.load_folder(d)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_request_grows_out_of_short_contexts(model, dtype):
    from swifttransformer_amd.engine.step import StepEntry
    from swifttransformer_amd.ops.tuning import tuning
    d, cfg, w = model
    short, n = tuning.short_span, 8
    first = short - 4                                # contexts of the decode steps: first + 1 .. first + n, across `short`
    seqs = [tiny.prompt(first + n, CFG["vocab_size"], 1), tiny.prompt(20 + n, CFG["vocab_size"], 2)]
    refs = [plain_opt.forward(cfg, w, s).numpy() for s in seqs]
    runner = make_runner(d, DTYPES[dtype], 16, num_pages=40, max_seqs=2)
    starts = [first, 20]
    for r, s in enumerate(seqs):
        runner.admit(r)
        runner.step([StepEntry(r, s[:starts[r]], [])])
    for k in range(n):
        logits = runner.step([StepEntry(r, [seqs[r][starts[r] + k]], [0]) for r in range(2)])
        check(logits, np.stack([refs[r][starts[r] + k] for r in range(2)]), DTYPES[dtype], f"{dtype} step {k}")
        want = short if first + k + 1 <= short else 1024
        assert runner._recorded[2] is runner._recorded_spans[2, want]
        assert runner._recorded[2].buffers.ctx.max_kv_len == want
    assert set(runner._recorded_spans) == {(2, short), (2, 1024)}


def test_tokens_chosen_on_the_device_cross_over(model):
    """Greedy decoding that runs a step ahead of the host: the next step's ids come from the other recording's best tokens."""
    from swifttransformer_amd.engine.engine import Engine
    from swifttransformer_amd.ops.tuning import tuning
    from swifttransformer_amd.sampling import SamplingParams
    d, cfg, w = model
    prompt = tiny.prompt(tuning.short_span - 5, CFG["vocab_size"], 9)
    eng = Engine(d, dtype="fp32", page_size=16, num_pages=40, max_seqs=2)
    out = eng.generate([prompt], SamplingParams(max_new_tokens=12, ignore_eos=True))[0]
    assert out == plain_opt.generate(cfg, w, prompt, 12)
    assert len(eng.runner._recorded_spans) == 2


def test_warm_up_records_both(model):
    from swifttransformer_amd.ops.tuning import tuning
    runner = make_runner(model[0], torch.float32, 16, num_pages=40, max_seqs=2)
    assert runner.warm_up([], [1, 2]) == 4
    assert set(runner._recorded_spans) == {(b, s) for b in (1, 2) for s in (tuning.short_span, 1024)}
    assert runner.warm_up([], [1, 2]) == 0


def test_models_no_longer_than_short_contexts_have_one(tmp_path):
    from swifttransformer_amd.engine.step import StepEntry
    from swifttransformer_amd.config import OptHyperParam
    from swifttransformer_amd.ops.tuning import tuning
    from swifttransformer_amd.weights import write_random_model
    d = write_random_model(OptHyperParam(**dict(CFG, max_position_embeddings=tuning.short_span)).validate(), str(tmp_path / "m"), seed=3)
    runner = make_runner(d, torch.float32, 16, num_pages=8, max_seqs=1)
    runner.admit(0)
    runner.step([StepEntry(0, [5], [0])])
    assert set(runner._recorded_spans) == {(1, tuning.short_span)}


def test_one_recording_where_the_step_is_the_same(tmp_path):
    """Fewer positions than two splits of keys: a request that grows out of short contexts keeps its recording."""
    from swifttransformer_amd.engine.step import StepEntry
    from swifttransformer_amd.config import OptHyperParam
    from swifttransformer_amd.ops.tuning import tuning
    from swifttransformer_amd.weights import write_random_model
    most = 2 * tuning.min_keys_per_split - 1
    d = write_random_model(OptHyperParam(**dict(CFG, max_position_embeddings=most)).validate(), str(tmp_path / "m"), seed=3)
    cfg, w = plain_opt.load_folder(d)
    runner = make_runner(d, torch.float32, 16, num_pages=40, max_seqs=2)
    seq, first = tiny.prompt(tuning.short_span + 3, CFG["vocab_size"], 5), tuning.short_span - 3
    ref = plain_opt.forward(cfg, w, seq).numpy()
    runner.admit(0)
    runner.step([StepEntry(0, seq[:first], [])])
    for p in range(first, len(seq)):
        check(runner.step([StepEntry(0, [seq[p]], [0])]), ref[p:p + 1], torch.float32, f"position {p}")
    assert set(runner._recorded_spans) == {(1, most)}
    runner.finish(0)
    assert runner.warm_up([], [1, 2]) == 1 and set(runner._recorded_spans) == {(1, most), (2, most)}
