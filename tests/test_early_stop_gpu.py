"""Generation that stops early: the loop that enqueues the next step's first layers before it knows
whether the step is needed, against the loop that asks after every step (graph mode).  Models that
end at once, after a few steps, and never; two calls each, since a step enqueued too far must
leave nothing behind."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eos", [0.0, 1.5, 3.0, 8.0])
@pytest.mark.parametrize("batch,method", [(1, "beam_search"), (3, "beam_search"), (2, "topk"),
                                          (2, "topk_greedy")])
def test_translate(tmp_path, batch, method, eos):
    from lightseq_amd import synthetic
    from lightseq_amd.inference import QuantTransformer
    cfg = synthetic.transformer_config("tiny")
    cfg.update(sampling_method=method, topk=4, topp=0.9)
    path = os.path.join(str(tmp_path), "qt.pb")
    synthetic.write_quant_transformer(path, cfg, seed=5, w_std=0.2,
                                      eos_bias=eos * 0.02 * np.sqrt(cfg["hidden"]))
    res = []
    for graphs in (False, True):
        model = QuantTransformer(path, 4)
        model.graph_mode(graphs)
        for seed in (1, 2):
            ids, _ = synthetic.make_token_ids(dict(vocab=cfg["src_vocab"], padding_id=cfg["padding_id"]),
                                              batch, 9, seed=seed)
            model.set_seed(7)
            tokens, scores = model.infer(ids)
            res.append((np.array(tokens), np.array(scores), model.steps_run()))
        model.close()
    for a, b in zip(res[:2], res[2:]):
        assert a[2] == b[2]
        np.testing.assert_array_equal(a[0], b[0])
        np.testing.assert_array_equal(a[1], b[1])


@pytest.mark.parametrize("eos", [0.0, 2.0, 8.0])
@pytest.mark.parametrize("batch,topk", [(1, 1), (3, 1), (2, 4)])
def test_generate(tmp_path, batch, topk, eos):
    from lightseq_amd import synthetic
    from lightseq_amd.inference import QuantGpt
    cfg = synthetic.gpt_config("tiny")
    cfg.update(topk=topk)
    path = os.path.join(str(tmp_path), "gpt.pb")
    synthetic.write_quant_gpt(path, cfg, seed=6, w_std=0.2)
    rng = np.random.default_rng(3)
    ids = [rng.integers(1, cfg["vocab"] - 2, size=(batch, 7), dtype=np.int32) for _ in range(2)]
    if eos:  # the id this model says first (after `eos` more tokens) ends a sequence
        model = QuantGpt(path, 4)
        cfg["eos_id"] = int(np.asarray(model.sample(ids[0]))[0, 7 + int(eos) - 2])
        model.close()
        synthetic.write_quant_gpt(path, cfg, seed=6, w_std=0.2)
    res = []
    for graphs in (False, True):
        model = QuantGpt(path, 4)
        model.graph_mode(graphs)
        for a in ids:
            model.set_seed(7)
            res.append((np.array(model.sample(a)), model.steps_run()))
        model.close()
    for a, b in zip(res[:2], res[2:]):
        assert a[1] == b[1]
        np.testing.assert_array_equal(a[0], b[0])
