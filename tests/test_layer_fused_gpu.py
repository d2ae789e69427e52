"""The fused launches of the quantised layers at the edges of their tiles: widths that are padded to
64 bytes, one row, key counts around the blocks of the attention kernels, every mask type; and the
same bits for a sequence whatever batch it is computed in, i.e. whichever kernel and tile the
products take."""
import numpy as np
import pytest
import torch

from helpers import DEV, to_dev, to_np
from test_decoder_layer_gpu import _case, _make_stack, _release
from test_layer_ops_gpu import _lo, _make_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,seq,hs,nh,ims,pre_ln,act,mask_type", [
    (1, 1, 96, 3, 208, False, "relu", torch.float32),
    (2, 33, 128, 2, 192, True, "gelu", torch.bool),
    (2, 129, 64, 1, 144, False, "gelu", torch.int64),
    (3, 65, 256, 2, 320, True, "relu", torch.float16),
    (1, 128, 160, 5, 64, False, "relu", torch.int32),
    (2, 17, 128, 4, 256, True, "relu", torch.float64),
])
def test_encoder_layer_edges(batch, seq, hs, nh, ims, pre_ln, act, mask_type):
    from test_oracle_layer_ops import config0
    rng = np.random.default_rng(seq)
    cfg0 = config0(rng, pre_ln, act, batch, seq, hs, nh, ims)
    layer, para = _make_layer(cfg0, pre_ln, act, nh, 512, 256)
    x = cfg0[1].astype(np.float16)
    pad = np.zeros((batch, seq), np.float32)
    pad[batch - 1, seq - seq // 3:] = 1
    with torch.no_grad():
        got = to_np(layer(to_dev(x), to_dev(pad).to(mask_type)))
    with np.errstate(over="ignore"):
        mask = (pad * -1e8).astype(np.float16)
    want = _lo().encoder_layer_forward(para, x, mask, nh, ims, pre_ln, act)
    d = np.abs(got.astype(np.float64) - want.astype(np.float64))
    assert d.max() < 2e-2 and d.mean() < 1e-3, (d.max(), d.mean())


@pytest.mark.parametrize("hs,ims,seq", [(512, 2048, 64), (768, 3072, 37), (768, 3072, 64), (768, 3072, 128),
                                        (1024, 4096, 61)])
def test_a_sequence_does_not_depend_on_its_batch(hs, ims, seq):
    from test_oracle_layer_ops import config0
    rng = np.random.default_rng(5)
    cfg0 = config0(rng, False, "relu", 60, seq, hs, hs // 64, ims)
    layer, _ = _make_layer(cfg0, False, "relu", hs // 64, 60 * seq, 128)
    x = to_dev(cfg0[1].astype(np.float16))
    pad = torch.zeros(60, seq, device=DEV)
    with torch.no_grad():
        full = layer(x, pad)
        for n in (1, 3, 9, 20):
            assert torch.equal(layer(x[:n].contiguous(), pad[:n].contiguous()), full[:n])


@pytest.mark.parametrize("hs,nh,trg,src", [(512, 8, 61, 20), (1024, 16, 31, 64)])
def test_a_target_does_not_depend_on_its_batch(hs, nh, trg, src):
    """The same of a decoder layer: products into heads and caches, residuals, keys and values of the
    encoder output, by tiles of 16 x 16 to 256 x 256 with remainders in rows."""
    from lightseq_amd import layers as L
    L.LSTransformerDecoderLayer.new_stack()
    torch.manual_seed(7)
    cfg = L.LSTransformerDecoderLayer.get_config(
        max_batch_tokens=80 * max(trg, src), max_seq_len=64, hidden_size=hs, intermediate_size=4 * hs, nhead=nh,
        attn_prob_dropout_ratio=0.0, activation_dropout_ratio=0.0, hidden_dropout_ratio=0.0, pre_layer_norm=True,
        fp16=True, local_rank=0, nlayer=1, activation_fn="relu")
    layer = L.LSTransformerDecoderLayer(cfg).half().to(DEV).eval()
    layer.enable_quant()
    at = layer.para_offset[18]
    n = layer.para_offset[19] - at
    with torch.no_grad():
        layer.para[at:at + n] = torch.tensor([4.0, 0.15, 6.0], dtype=torch.half, device=DEV).repeat(n // 3)
    try:
        x = torch.randn(80, trg, hs, device=DEV).half()
        enc = torch.randn(src, 80, hs, device=DEV).half()
        pad = torch.zeros(80, src, device=DEV)
        with torch.no_grad():
            full = layer(x, enc, pad)
            for b in (1, 2, 7, 16, 33):
                got = layer(x[:b].contiguous(), enc[:, :b].contiguous(), pad[:b].contiguous())
                assert torch.equal(got, full[:b]), b
    finally:
        _release([layer])


@pytest.mark.parametrize("trg,src,pre_ln", [(1, 1, False), (33, 64, True), (64, 33, False)])
def test_decoder_layer_edges(trg, src, pre_ln):
    """The encoder output as a transposed view and as a tensor of its own give the same bits, and
    both agree with the restatement."""
    lo = _lo()
    paras, x, enc, pad, mask = _case(trg, 2, trg, src)
    layers = _make_stack(paras, pre_ln, "relu", 128, 64)
    try:
        from test_decoder_layer_gpu import IMS, NH, NLAYER
        kv = lo.decoder_encdec_kv(paras[0], enc, NH, IMS, NLAYER)
        enc_t = to_dev(enc).transpose(0, 1)
        for lid, layer in enumerate(layers):
            with torch.no_grad():
                got = layer(to_dev(x), enc_t, to_dev(pad).bool())
                assert torch.equal(layer(to_dev(x), enc_t.contiguous(), to_dev(pad)), got)
            want = lo.decoder_layer_forward(paras[lid], lid, NLAYER, x, kv, mask, NH, IMS, pre_ln, "relu")
            d = np.abs(to_np(got).astype(np.float64) - want.astype(np.float64))
            assert d.max() < 2e-2 and d.mean() < 1e-3, (lid, d.max(), d.mean())
    finally:
        _release(layers)
