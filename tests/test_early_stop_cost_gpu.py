"""What a generation run that ends early computes for nothing: one layer per step it made at most, of
deep models whose steps are mostly layers.  Times between events on the model's stream, the
smallest of several runs."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS = 32


def _steps_ms(model, call, reps=15):
    """(time of the step loop, steps of the loop) of the fastest of `reps` calls."""
    call()
    best = None
    for _ in range(reps):
        call()
        _, ms, steps = model.phase_times()
        best = ms if best is None else min(best, ms)
    return best, steps


def test_translate(tmp_path):
    """Two steps and two layers against the average step of a run that does not end early: 1.7 of them
    (the first step has less to read), where a whole step enqueued ahead made 2.6."""
    from lightseq_amd import synthetic
    from lightseq_amd.inference import QuantTransformer
    cfg = synthetic.transformer_config("tiny")
    cfg.update(n_enc_layer=1, n_dec_layer=LAYERS)
    path = os.path.join(str(tmp_path), "qt.pb")
    ids, _ = synthetic.make_token_ids(dict(vocab=cfg["src_vocab"], padding_id=cfg["padding_id"]), 1, 9, seed=1)
    ms = {}
    for name, eos in (("long", -4.0), ("short", 20.0)):
        synthetic.write_quant_transformer(path, cfg, seed=5, eos_bias=eos * 0.02 * np.sqrt(cfg["hidden"]))
        model = QuantTransformer(path, 1)
        ms[name] = _steps_ms(model, lambda: model.infer(ids))
        model.close()
    assert ms["short"][1] == 2 and ms["long"][1] >= 8, ms
    per_step = ms["long"][0] / ms["long"][1]
    assert ms["short"][0] < 2.1 * per_step, ms


def test_generate(tmp_path):
    """A text that ends with its first token (no step, one layer) against one that ends with its
    second (one step, two layers): 0.03 of its time, where three quarters of a step ahead made 0.42."""
    from lightseq_amd import synthetic
    from lightseq_amd.inference import QuantGpt
    cfg = synthetic.gpt_config("tiny")
    cfg.update(n_layer=LAYERS, topk=1)
    path = os.path.join(str(tmp_path), "gpt.pb")
    ids = np.random.default_rng(3).integers(1, cfg["vocab"] - 2, size=(1, 7), dtype=np.int32)
    synthetic.write_quant_gpt(path, cfg, seed=6, w_std=0.2)
    model = QuantGpt(path, 1)
    text = np.asarray(model.sample(ids))[0, 7:].tolist()
    model.close()
    assert text[0] != text[1]
    ms = []
    for n in (0, 1):
        cfg["eos_id"] = int(text[n])
        synthetic.write_quant_gpt(path, cfg, seed=6, w_std=0.2)
        model = QuantGpt(path, 1)
        ms.append(_steps_ms(model, lambda: model.sample(ids)))
        assert model.steps_run() == n + 1
        model.close()
    assert [s for _, s in ms] == [0, 1], ms
    assert ms[0][0] < 0.2 * ms[1][0], ms
