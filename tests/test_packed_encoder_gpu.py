"""The encoder without its padding rows leaves the bytes of the padded route (the one taps select),
wherever the padding is and whether the host knows the ids or waits for the plan."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    from lightseq_amd import inference, synthetic
    cfg = dict(synthetic.bert_config("bert_base"), n_layer=2, vocab=500, max_step=320)
    path = os.path.join(str(tmp_path_factory.mktemp("pack")), "m.pb")
    synthetic.write_quant_bert(path, cfg, seed=3)
    m = inference.QuantBert(path, 20)
    m.cfg = cfg
    yield m
    m.close()


def _ids(cfg, lens, seq, holes=()):
    rng = np.random.default_rng(len(lens) * seq)
    ids = rng.integers(1, cfg["vocab"], size=(len(lens), seq), dtype=np.int32)
    ids[np.arange(seq)[None, :] >= np.asarray(lens)[:, None]] = cfg["padding_id"]
    for b, s in holes:
        ids[b, s] = cfg["padding_id"]
    return ids


@pytest.mark.parametrize("lens,seq,holes", [
    ([1], 1, []), ([17], 17, []), ([5], 40, []), ([40, 33, 1, 64], 64, [(0, 0), (1, 7), (3, 62)]),
    ([0, 128, 31, 32, 33, 0, 65, 127], 128, []), ([96] * 8, 96, []), ([0, 0], 20, []),
    ([129, 1, 130], 130, [(2, 64)]), ([300, 0, 128, 129, 257], 300, [(0, 100)]), ([3, 9, 11, 2, 7] * 4, 12, [])])
def test_same_bytes_as_the_padded_route(model, lens, seq, holes):
    ids = _ids(model.cfg, lens, seq, holes)
    packed_host = model.infer_fp16(ids)
    d_ids = torch.from_numpy(ids).to(DEV)
    model.set_input_ptr(0, d_ids.data_ptr())
    model.set_input_shape(0, ids.shape)
    model.infer_device()
    packed_device = model._download(0).cpu().numpy()
    tap = torch.zeros(ids.size * model.cfg["hidden"], dtype=torch.int8, device=DEV)
    model.set_tap(0, "ctx_q", tap)
    padded = model.infer_fp16(ids)
    model.set_tap(0, "ctx_q", None)
    np.testing.assert_array_equal(packed_host.view(np.uint16), padded.view(np.uint16))
    np.testing.assert_array_equal(packed_device.view(np.uint16), padded.view(np.uint16))
