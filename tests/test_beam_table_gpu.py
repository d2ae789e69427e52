"""Beam search over caches whose rows stay where they were computed (a table says which beam's row
holds a step) against the same run with the rows moved after every step: the route of runs that
record their steps.  Every form of the attention kernel: four pairs a workgroup, one pair over up
to 256 steps, wide groups beyond, several rounds of loads."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# 1030 steps of heads of 128 do not fit one round of the widest group (512)
@pytest.mark.parametrize("hidden,heads,beam,max_step,batch,seed", [
    (128, 4, 4, 32, 3, 1), (128, 2, 2, 90, 2, 2), (256, 2, 8, 150, 2, 3), (128, 2, 4, 300, 2, 4),
    (128, 4, 1, 40, 2, 5), (256, 2, 4, 560, 1, 6), (128, 1, 32, 41, 1, 7),
])
def test_tokens_and_scores_of_the_run_that_moves_rows(tmp_path, hidden, heads, beam, max_step, batch, seed):
    from lightseq_amd import inference, synthetic
    cfg = dict(synthetic.transformer_config("tiny"), hidden=hidden, head_num=heads, inner=128, beam_size=beam,
               max_step=max_step, extra_decode_length=max_step)
    path = os.path.join(str(tmp_path), "m.pb")
    sigma = 0.02 * np.sqrt(hidden)
    synthetic.write_quant_transformer(path, cfg, seed=seed, eos_bias=0.5 * sigma, w_std=0.2)
    ids = np.random.default_rng(seed).integers(4, cfg["src_vocab"], size=(batch, 9), dtype=np.int32)
    model = inference.QuantTransformer(path, batch)
    try:
        tokens, scores = model.infer(ids)
        steps = model.steps_run()
        again = model.infer(ids)  # tables left over from a call do not matter
        np.testing.assert_array_equal(again[0], tokens)
        rows = batch * beam
        rec = torch.zeros(max_step, rows, max_step, dtype=torch.int32, device="cuda")
        model.set_step_record(None, rec, max_step)
        moved_tokens, moved_scores = model.infer(ids)
        assert model.steps_run() == steps and steps > max_step // 3
        np.testing.assert_array_equal(moved_tokens, tokens)
        np.testing.assert_array_equal(moved_scores, scores)
        model.set_step_record(None, None, 0)
        model.graph_mode(True)
        for _ in range(3):
            np.testing.assert_array_equal(model.infer(ids)[0], tokens)
        alive = rec[:steps].cpu().numpy()
    finally:
        model.close()
    if beam > 1:  # beams did change places
        changed = sum(int((alive[s, :, :s + 1] != alive[s - 1, :, :s + 1]).any()) for s in range(1, steps))
        assert changed > steps // 8, changed
