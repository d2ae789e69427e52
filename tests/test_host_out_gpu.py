"""The output memory of ls_model_infer_host: a kernel writes it, so it has to be pinned."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_ordinary_memory_is_refused(tmp_path):
    from lightseq_amd import inference, lib, synthetic
    cfg = synthetic.bert_config("tiny")
    path = os.path.join(str(tmp_path), "tiny.pb")
    synthetic.write_quant_bert(path, cfg, seed=0)
    model = inference.QuantBert(path, 4)
    try:
        ids, _ = synthetic.make_token_ids(cfg, 3, 40, seed=1)
        want = model.infer(ids)
        for f16, dtype in ((False, np.float32), (True, np.float16)):
            plain = np.full(want.shape, 7, dtype)
            with pytest.raises(lib.LSHError, match="not pinned"):
                model._infer_host(ids, plain, f16)
            assert (plain == 7).all()
            # nothing is left behind: neither a pending error nor a changed model
            pinned = torch.zeros(want.shape, dtype=torch.float16 if f16 else torch.float32, pin_memory=True).numpy()
            torch.zeros(4, device="cuda").add_(1).cpu()
            model._infer_host(ids, pinned, f16)
            np.testing.assert_array_equal(pinned, want.astype(dtype))
    finally:
        model.close()


def _ragged(lens, seq, pad, rng):
    ids = rng.integers(1, 90, size=(len(lens), seq), dtype=np.int32)
    for b, n in enumerate(lens):
        ids[b, n:] = pad
        if n > 3:
            ids[b, 1] = pad  # padding inside a sequence is one of its rows
    return ids


@pytest.mark.parametrize("name,lens,seq", [
    ("bert_base", [384] * 3 + [1, 0, 200, 383, 64, 97], 384),  # 1.1 MB of padding and more: sent ahead
    ("bert_base", [128, 20, 3] + [90] * 29, 128),
    ("bert_base", [0, 0, 0], 512),
    ("bert_base", [512, 171], 512),  # one position of padding short of 1 MiB in floats
    ("bert_base", [512, 170], 512),
])
def test_padding_sent_ahead_is_the_padding_of_the_stack(tmp_path_factory, name, lens, seq):
    """Result by host memory against the one that stays on the device, in both formats."""
    from lightseq_amd import inference, synthetic
    cfg = dict(synthetic.bert_config(name), n_layer=2, vocab=128)
    path = os.path.join(str(tmp_path_factory.mktemp("pads")), "m.pb")
    synthetic.write_quant_bert(path, cfg, seed=3)
    model = inference.QuantBert(path, 32)
    try:
        ids = _ragged(lens, seq, cfg["padding_id"], np.random.default_rng(seq))
        dev = torch.from_numpy(ids).cuda()
        out = torch.zeros(len(lens), seq, cfg["hidden"], dtype=torch.half, device="cuda")
        model.infer(ids[:1])  # another shape first
        got32, got16 = model.infer(ids).copy(), model.infer_fp16(ids).copy()
        plain = inference.LSModel("QuantBert", path, 32)
        try:
            plain.set_input_ptr(0, dev.data_ptr())
            plain.set_input_shape(0, dev.shape)
            plain.set_output_ptr(0, out.data_ptr())
            plain.infer_device()
            want = out.cpu().numpy()
        finally:
            plain.close()
        np.testing.assert_array_equal(got16, want)
        np.testing.assert_array_equal(got32, want.astype(np.float32))
    finally:
        model.close()
