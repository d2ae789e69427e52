"""Decoder attention launches that go through the out-projection, int32 sums requantised by the layer
norm behind, against the same steps with products of their own (a set tap keeps them apart): the
same logits and tokens, eager and replayed from graphs.  Caches around every change of the kernel's form (64,
128, 256, 512, 640 and beyond 1024 steps, where the launch ends), one to more rows than a
workgroup takes, batches that outgrow one round of the chip on the way."""
import os

import numpy as np
import pytest
import torch

from helpers import DEV

pytestmark = pytest.mark.gpu


def _run(kind, path, cfg, ids, tapped):
    from lightseq_amd import inference
    model = getattr(inference, kind)(path, ids.shape[0])
    rows = ids.shape[0] * cfg.get("beam_size", 1)
    vocab = cfg.get("trg_vocab", cfg.get("vocab"))
    most = cfg["max_step"] if kind != "QuantGpt" else cfg["extra_decode_length"] + 2
    call = (lambda: (model.sample(ids),)) if kind == "QuantGpt" else (lambda: model.infer(ids))
    try:
        model.benchmark_mode(True)
        tap = torch.zeros(rows, cfg["hidden"], dtype=torch.int8, device=DEV)
        if tapped:
            model.set_tap(0, "dec.next_ln_q", tap)
            model.set_tap_step(1)
        logits = torch.zeros(most, rows, vocab, dtype=torch.int8, device=DEV)
        if kind == "QuantGpt":
            model.set_step_record(logits, most)
        else:
            model.set_step_record(logits, None, most)
        out = [[np.asarray(o) for o in call()]]
        steps = model.steps_run()
        assert steps <= most
        model.set_step_record(*([None, 0] if kind == "QuantGpt" else [None, None, 0]))
        if not tapped:
            out += [[np.asarray(o) for o in call()]]
            model.graph_mode(True)
            for _ in range(2):
                out += [[np.asarray(o) for o in call()]]
        return out, logits[:steps].cpu().numpy()
    finally:
        model.close()


def _same(kind, path, cfg, ids, first=None):
    want, want_logits = _run(kind, path, cfg, ids, True)
    got, got_logits = _run(kind, path, cfg, ids, False)
    np.testing.assert_array_equal(want_logits, got_logits)
    assert want_logits.any()
    for run in got[:first]:
        for a, b in zip(want[0], run):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("batch,hidden,prompt,extra", [
    (1, 256, 3, 12), (2, 384, 61, 6), (3, 1024, 62, 5), (4, 128, 125, 6), (5, 1024, 126, 6), (16, 1024, 253, 6),
    (7, 512, 508, 6), (1, 768, 639, 4), (1, 1024, 1021, 7), (64, 1024, 126, 6), (33, 1024, 9, 4),
])
def test_gpt_steps(tmp_path, batch, hidden, prompt, extra):
    from lightseq_amd import synthetic
    cfg = synthetic.gpt_config("tiny")
    cfg.update(hidden=hidden, inner=2 * hidden, head_num=hidden // 64, vocab=97, eos_id=96, n_layer=2,
               max_step=prompt + extra + 1, extra_decode_length=extra)
    path = os.path.join(str(tmp_path), "gpt.pb")
    synthetic.write_quant_gpt(path, cfg, seed=3, w_std=0.2)
    rng = np.random.default_rng(batch)
    _same("QuantGpt", path, cfg, rng.integers(1, 95, size=(batch, prompt), dtype=np.int32))


@pytest.mark.parametrize("batch,beam,hidden,seq,extra,gelu,post", [
    (1, 4, 256, 9, 12, False, False), (3, 1, 768, 31, 70, True, True), (2, 2, 512, 100, 40, False, False),
    (5, 4, 1024, 17, 10, False, True), (16, 4, 1024, 20, 130, False, False),
    (1, 4, 512, 130, 12, False, False),  # a long source: the cross attention apart
    (2, 4, 384, 12, 30, True, False),    # its layer norm apart
    (2, 8, 512, 7, 12, False, False),    # more beams than its launch covers
    (40, 1, 1024, 7, 6, False, False),   # more sentences than one round
])
def test_decoder_steps(tmp_path, batch, beam, hidden, seq, extra, gelu, post):
    from lightseq_amd import synthetic
    cfg = synthetic.transformer_config("tiny")
    cfg.update(hidden=hidden, inner=2 * hidden, head_num=hidden // 64, beam_size=beam, use_gelu=gelu,
               is_post_ln=post, max_step=max(160, seq + extra), extra_decode_length=extra)
    path = os.path.join(str(tmp_path), "qt.pb")
    synthetic.write_quant_transformer(path, cfg, seed=4, w_std=0.2)
    ids, _ = synthetic.make_token_ids(dict(vocab=cfg["src_vocab"], padding_id=cfg["padding_id"]), batch,
                                      seq, seed=batch)
    _same("QuantTransformer", path, cfg, ids)


@pytest.mark.parametrize("method", ["topk", "topp", "topk_greedy"])
def test_decoder_steps_that_sample(tmp_path, method):
    from lightseq_amd import synthetic
    cfg = synthetic.transformer_config("tiny")
    cfg.update(hidden=512, inner=256, head_num=8, sampling_method=method, topk=4, topp=0.8, beam_size=4,
               max_step=64, extra_decode_length=20)
    path = os.path.join(str(tmp_path), "qt.pb")
    synthetic.write_quant_transformer(path, cfg, seed=6, w_std=0.2)
    ids = np.random.default_rng(5).integers(4, cfg["src_vocab"], size=(3, 11), dtype=np.int32)
    _same("QuantTransformer", path, cfg, ids, first=1)  # (later calls draw other numbers)


# batches of few positions and beyond the limit: a workgroup's share of the columns (8 .. 1 blocks of 16 a wavefront),
# one to three blocks of 32 tokens, sequences of nothing but padding, holes
@pytest.mark.parametrize("hidden,lens,seq,holes", [
    (128, [1], 1, []), (256, [17, 3], 17, []), (768, [16], 16, []), (768, [5], 40, []), (1024, [33, 0, 40], 40, [(0, 2)]),
    (512, [64, 63], 64, [(1, 7)]), (768, [96], 96, []), (768, [97], 97, []), (1024, [128], 128, [(0, 64)]), (768, [0, 0], 20, []),
    (768, [3, 9, 11, 2, 7] * 2, 12, []), (1024, [1, 2, 0, 4] * 8, 4, []), (384, [65], 70, []),
])
@pytest.mark.parametrize("post", [False, True])
def test_encoder(tmp_path, hidden, lens, seq, holes, post):
    from lightseq_amd import inference, synthetic
    cfg = dict(synthetic.bert_config("tiny"), n_layer=3, hidden=hidden, inner=2 * hidden, head_num=hidden // 64,
               vocab=300, max_step=128, is_post_ln=post)
    path = os.path.join(str(tmp_path), "m.pb")
    synthetic.write_quant_bert(path, cfg, seed=3)
    ids = np.random.default_rng(seq).integers(1, cfg["vocab"], size=(len(lens), seq), dtype=np.int32)
    ids[np.arange(seq)[None, :] >= np.asarray(lens)[:, None]] = cfg["padding_id"]
    for b, s in holes:
        ids[b, s] = cfg["padding_id"]
    model = inference.QuantBert(path, len(lens))
    try:
        got = [model.infer_fp16(ids) for _ in range(2)]
        d_ids = torch.from_numpy(ids).to(DEV)
        model.set_input_ptr(0, d_ids.data_ptr())
        model.set_input_shape(0, ids.shape)
        model.infer_device()
        got.append(model._download(0).cpu().numpy())
        tap = torch.zeros(ids.size * hidden, dtype=torch.int8, device=DEV)
        model.set_tap(0, "ctx_q", tap)  # the route with products of their own
        want = model.infer_fp16(ids)
        for g in got:
            np.testing.assert_array_equal(g.view(np.uint16), want.view(np.uint16))
    finally:
        model.close()
