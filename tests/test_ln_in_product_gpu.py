"""Generation steps whose layer norms are made by the products that read them (and by the
cross-attention launch) against the same steps with launches of their own: the same logits and
tokens, over the row counts and widths the rule covers and their edges.  A set tap keeps the
launches apart."""
import os

import numpy as np
import pytest
import torch

from helpers import DEV

pytestmark = pytest.mark.gpu


def _run(kind, path, cfg, ids, tapped):
    from lightseq_amd import inference
    model = getattr(inference, kind)(path, ids.shape[0])
    model.benchmark_mode(True)
    rows = ids.shape[0] * cfg.get("beam_size", 1)
    vocab = cfg.get("trg_vocab", cfg.get("vocab"))
    logits = torch.zeros(cfg["max_step"], rows, vocab, dtype=torch.int8, device=DEV)
    tap = torch.zeros(rows, cfg["hidden"], dtype=torch.int8, device=DEV)
    if kind == "QuantGpt":
        model.set_step_record(logits, cfg["max_step"])
    else:
        alive = torch.zeros(cfg["max_step"], rows, cfg["max_step"], dtype=torch.int32, device=DEV)
        model.set_step_record(logits, alive, cfg["max_step"])
    if tapped:
        model.set_tap(0, "dec.next_ln_q", tap)
        model.set_tap_step(1)
    out = model.sample(ids) if kind == "QuantGpt" else model.infer(ids)[0]
    steps = model.steps_run()
    model.close()
    return np.asarray(out), logits[:steps].cpu().numpy()


def _same(kind, path, cfg, ids):
    want, want_logits = _run(kind, path, cfg, ids, True)
    got, got_logits = _run(kind, path, cfg, ids, False)
    np.testing.assert_array_equal(want_logits, got_logits)
    np.testing.assert_array_equal(want, got)


@pytest.mark.parametrize("batch,hidden,vocab", [(1, 256, 97), (2, 512, 128), (3, 768, 130),
                                                (4, 1024, 257), (5, 512, 97), (1, 320, 97)])
def test_gpt_steps(tmp_path, batch, hidden, vocab):
    from lightseq_amd import synthetic
    cfg = synthetic.gpt_config("tiny")
    cfg.update(hidden=hidden, inner=4 * hidden, head_num=hidden // 64, vocab=vocab, eos_id=vocab - 1,
               n_layer=3)
    path = os.path.join(str(tmp_path), "gpt.pb")
    synthetic.write_quant_gpt(path, cfg, seed=3, w_std=0.2)
    rng = np.random.default_rng(batch)
    _same("QuantGpt", path, cfg, rng.integers(1, vocab - 2, size=(batch, 6), dtype=np.int32))


@pytest.mark.parametrize("batch,beam,hidden,head,seq,gelu,post", [
    (1, 4, 256, 64, 9, False, False), (1, 2, 512, 64, 31, True, True), (3, 1, 768, 64, 17, False, True),
    (4, 4, 1024, 64, 5, False, False),   # only the cross-attention launch makes its layer norm
    (1, 4, 512, 32, 12, True, False),    # query product and attention apart
    (2, 8, 512, 64, 7, False, False),    # more beams than either covers
])
def test_decoder_steps(tmp_path, batch, beam, hidden, head, seq, gelu, post):
    from lightseq_amd import synthetic
    cfg = synthetic.transformer_config("tiny")
    cfg.update(hidden=hidden, inner=4 * hidden, head_num=hidden // head, beam_size=beam, use_gelu=gelu,
               is_post_ln=post)
    path = os.path.join(str(tmp_path), "qt.pb")
    synthetic.write_quant_transformer(path, cfg, seed=4, w_std=0.2)
    ids, _ = synthetic.make_token_ids(dict(vocab=cfg["src_vocab"], padding_id=cfg["padding_id"]), batch,
                                      seq, seed=batch)
    _same("QuantTransformer", path, cfg, ids)
