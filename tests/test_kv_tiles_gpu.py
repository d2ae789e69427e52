"""The projection of an encoder output to all layers' keys and values in tiles of 256 x 192 and 256 x 256
(976 and 1200 rows of 12288 columns, ragged in both) against the same sentences a few at a time, in
small tiles (checked against the oracle elsewhere): every output is one chain of products in ascending K,
so the bits do not depend on the tile."""
import os

import numpy as np
import pytest
import torch

from helpers import DEV

pytestmark = pytest.mark.gpu


def _keys_values(path, cfg, ids, layer):
    from lightseq_amd import inference
    model = inference.QuantTransformer(path, ids.shape[0])
    try:
        model.benchmark_mode(True)
        bufs = {n: torch.zeros(ids.size * cfg["hidden"], dtype=torch.float16, device=DEV)
                for n in ("encdec_k", "encdec_v")}
        enc = torch.zeros(ids.size, cfg["hidden"], dtype=torch.float16, device=DEV)
        for n, b in bufs.items():
            model.set_tap(layer, "dec." + n, b)
        model.set_tap(-1, "enc_out", enc)
        model.set_tap_step(0)
        model.infer(ids)
        return [bufs[n].cpu().numpy().reshape(ids.shape[0], -1) for n in ("encdec_k", "encdec_v")], enc.cpu().numpy()
    finally:
        model.close()


@pytest.mark.parametrize("batch,seq", [(16, 61), (20, 60)])
def test_large_tiles_leave_the_bits_of_small_ones(tmp_path, batch, seq):
    from lightseq_amd import synthetic
    cfg = synthetic.transformer_config("tiny")
    cfg.update(hidden=512, inner=128, head_num=8, n_enc_layer=1, n_dec_layer=12, max_step=64, beam_size=1,
               extra_decode_length=1)
    path = os.path.join(str(tmp_path), "m.pb")
    synthetic.write_quant_transformer(path, cfg, seed=9, w_std=0.1)
    rng = np.random.default_rng(batch)
    ids = rng.integers(4, cfg["src_vocab"], size=(batch, seq), dtype=np.int32)
    for layer in (0, 11):
        big, enc = _keys_values(path, cfg, ids, layer)
        few, enc_few = _keys_values(path, cfg, ids[-2:], layer)
        np.testing.assert_array_equal(enc[-2 * seq:].view(np.uint16), enc_few.view(np.uint16))
        for a, b in zip(big, few):
            assert np.abs(b.astype(np.float32)).max() > 0
            np.testing.assert_array_equal(a[-2:].view(np.uint16), b.view(np.uint16))
        first, _ = _keys_values(path, cfg, ids[:2], layer)
        for a, b in zip(big, first):
            np.testing.assert_array_equal(a[:2].view(np.uint16), b.view(np.uint16))
