"""Perplexity of a batch of ragged texts, whose padded positions have no rows: every text's value is
the one it has alone, from host ids and from device ids."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    from lightseq_amd import synthetic
    from lightseq_amd.inference import QuantGpt
    import test_gpt_gpu as tg
    cfg = synthetic.gpt_config("tiny")
    cfg.update(sampling_method="ppl", hidden=128, inner=256, head_num=2, max_step=320)
    path, _ = tg._make(tmp_path_factory.mktemp("text"), cfg, 3, w_std=0.2)
    m = QuantGpt(path, 5)
    yield m, cfg
    m.close()


@pytest.mark.parametrize("seq,lens", [(17, (17, 1, 2, 16, 0)), (129, (129, 128, 5, 127)), (300, (300,)),
                                      (260, (0, 257, 64)), (9, (0, 0))])
def test_texts_alone_and_together(model, seq, lens):
    m, cfg = model
    rng = np.random.default_rng(seq)
    ids = np.full((len(lens), seq), cfg["padding_id"], np.int32)
    for b, n in enumerate(lens):
        ids[b, :n] = rng.integers(1, cfg["vocab"], n)
        ids[b, :n][ids[b, :n] == cfg["padding_id"]] = (cfg["padding_id"] + 1) % cfg["vocab"]
    got = m.ppl(ids)
    want = [m.ppl(ids[b:b + 1, :n])[0] if n > 1 else 0.0 for b, n in enumerate(lens)]
    # the rows of a product of another size are added in the same order: integers
    np.testing.assert_allclose(got, want, rtol=1e-6)
    dev = torch.from_numpy(ids).cuda()
    out = torch.full((len(lens),), 7.0, device="cuda")
    torch.cuda.synchronize()  # the model has a stream of its own
    m.set_input_ptr(0, dev.data_ptr())
    m.set_input_shape(0, list(ids.shape))
    own = m.get_output_ptr(0)
    m.set_output_ptr(0, out.data_ptr())
    m.infer_device()
    m.set_output_ptr(0, own)
    np.testing.assert_array_equal(out.cpu().numpy(), got)


def test_padding_inside_a_text(model):
    """A padding id between tokens keeps its row; the length is the number of tokens."""
    m, cfg = model
    rng = np.random.default_rng(1)
    ids = rng.integers(1, cfg["vocab"], (2, 20)).astype(np.int32)
    ids[ids == cfg["padding_id"]] = (cfg["padding_id"] + 1) % cfg["vocab"]
    ids[0, 4:6] = cfg["padding_id"]
    alone = m.ppl(ids[:1])
    assert np.isfinite(alone).all()
    np.testing.assert_allclose(m.ppl(ids)[0], alone[0], rtol=1e-6)
