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
