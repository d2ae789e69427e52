"""Host memory in, host memory out: the copies the model makes itself and the pinned results."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    from lightseq_amd import inference, synthetic
    cfg = synthetic.bert_config("tiny")
    path = os.path.join(str(tmp_path_factory.mktemp("io")), "tiny.pb")
    synthetic.write_quant_bert(path, cfg, seed=0)
    m = inference.QuantBert(path, 4)
    m.cfg = cfg
    yield m
    m.close()


@pytest.mark.parametrize("batch,seq", [(1, 1), (1, 3), (3, 5), (2, 31), (4, 64)])
def test_host_results_are_the_device_results(model, batch, seq):
    """Id counts with and without a remainder of the 16-byte copies; float32 and fp16 results."""
    import torch
    from lightseq_amd import synthetic
    ids, _ = synthetic.make_token_ids(model.cfg, batch, seq, seed=batch)
    f32, f16 = model.infer(ids), model.infer_fp16(ids)
    d_ids = torch.from_numpy(ids).cuda()
    model.set_input_ptr(0, d_ids.data_ptr())
    model.infer_device()
    want = model._download(0).cpu().numpy()
    assert f32.dtype == np.float32 and f16.dtype == np.float16
    np.testing.assert_array_equal(f16, want)
    np.testing.assert_array_equal(f32, want.astype(np.float32))


def test_kept_results_stay_and_the_pool_is_bounded(model):
    """Results that a caller keeps are never written again; beyond the pool's size they go to
    ordinary memory, and buffers come back when the results are dropped."""
    from lightseq_amd import synthetic
    batches = [synthetic.make_token_ids(model.cfg, 4, 64, seed=s)[0] for s in range(8)]
    kept = [model.infer(b) for b in batches]
    copies = [k.copy() for k in kept]
    assert len({k.ctypes.data for k in kept}) == len(kept)
    for k, c, b in zip(kept, copies, batches):
        np.testing.assert_array_equal(k, c)
        np.testing.assert_array_equal(k, model.infer(b))
    part = kept[0][1:, ::2]  # a view keeps its buffer
    want = part.copy()
    del kept, k
    for b in batches:
        model.infer(b)
    np.testing.assert_array_equal(part, want)
    assert model._results._left >= 0
