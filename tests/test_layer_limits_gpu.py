"""The quantised layers at the ends of what they accept: elements that are no finite numbers, rows
wider than a wavefront's registers, encoder outputs at odd places."""
import numpy as np
import pytest
import torch

from helpers import to_dev, to_np
from test_decoder_layer_gpu import IMS, NH, NLAYER, _case, _make_stack, _release
from test_layer_ops_gpu import _lo, _make_layer

pytestmark = pytest.mark.gpu

INF = np.float16(np.inf)


def _check(got, want, rows, bar=2e-2):
    """Outputs of the finite rows, within the bar of the layer tests."""
    got, want = to_np(got).astype(np.float64)[rows], want.astype(np.float64)[rows]
    assert np.isfinite(want).all()
    assert np.isfinite(got).all()
    d = np.abs(got - want)
    assert d.max() < bar and d.mean() < 1e-3, (d.max(), d.mean())


@pytest.mark.parametrize("pre_ln,act", [(False, "relu"), (False, "gelu"), (True, "relu"), (True, "gelu")])
@pytest.mark.parametrize("seq", [17, 150])
def test_infinite_elements_take_the_outermost_codes(pre_ln, act, seq):
    """Infinite weights, biases and (where the layer quantises its input itself) inputs have the
    codes +-127, as the restatement has them: every row but the infinite ones stays what it is.
    17 keys run the attention kernel of few queries, 150 the one of long sequences."""
    from test_oracle_layer_ops import config0
    lo = _lo()
    rng = np.random.default_rng(seq)
    batch, hs, nh, ims = 2, 128, 2, 256
    cfg0 = config0(rng, pre_ln, act, batch, seq, hs, nh, ims)
    layer, para = _make_layer(cfg0, pre_ln, act, nh, 512, 256)
    p = lo.split_params(para, hs, ims)  # views
    p["attn_qkvw"][hs + 3, 5], p["attn_qkvw"][2 * hs + 9, 7] = INF, -INF  # a key's and a value's row
    p["attn_qkvb"][2 * hs + 11] = -INF  # a column of the context
    p["attn_ow"][4, 6] = INF
    p["inter_w"][8, 2], p["inter_b"][10], p["inter_b"][12] = -INF, INF, np.float16(6e4)
    p["output_w"][1, 3], p["output_w"][2, 10] = INF, -INF
    with torch.no_grad():
        layer.para.copy_(to_dev(para))
    x = cfg0[1].astype(np.float16)
    rows = np.ones((batch, seq), bool)
    if not pre_ln:
        x[0, 4, 5], x[1, 16, 7], x[1, 2, 90] = INF, -INF, INF
        rows[0, 4] = rows[1, 16] = rows[1, 2] = False
    with np.errstate(all="ignore"):
        want = lo.encoder_layer_forward(para, x, np.zeros((batch, seq), np.float16), nh, ims, pre_ln, act)
    with torch.no_grad():
        got = layer(to_dev(x), torch.zeros(batch, seq, device="cuda"))
    _check(got, want, rows)


@pytest.mark.parametrize("act", ["relu", "gelu"])
def test_a_nan_has_the_code_of_minus_infinity(act):
    """Input or weight: the lesser bound, so that rows without one have the same bits either way."""
    from test_oracle_layer_ops import config0
    lo = _lo()
    batch, seq, hs, nh, ims = 2, 17, 128, 2, 256
    layer, para = _make_layer(config0(np.random.default_rng(4), False, act, batch, seq, hs, nh, ims), False, act, nh,
                              512, 256)
    x = config0(np.random.default_rng(5), False, act, batch, seq, hs, nh, ims)[1].astype(np.float16)
    outs = []
    for value in (np.float16(np.nan), -INF):
        q = para.copy()
        p = lo.split_params(q, hs, ims)
        p["attn_qkvw"][hs + 3, 5] = p["attn_ow"][4, 6] = p["inter_w"][8, 2] = p["output_w"][1, 3] = value
        y = x.copy()
        y[0, 4, 5] = y[1, 16, 7] = value
        with torch.no_grad():
            layer.para.copy_(to_dev(q))
            outs.append(to_np(layer(to_dev(y), torch.zeros(batch, seq, device="cuda"))))
    rows = np.ones((batch, seq), bool)
    rows[0, 4] = rows[1, 16] = False
    assert np.isfinite(outs[0][rows]).all() and not np.isfinite(outs[0][~rows]).any()
    np.testing.assert_array_equal(outs[0][rows], outs[1][rows])


def test_infinite_elements_of_a_decoder_layer():
    """The same with keys and values that the layer fake-quantises for its cache."""
    lo = _lo()
    paras, x, enc, pad, mask = _case(21, 2, 9, 12)
    for lid, para in enumerate(paras):
        p = lo.split_decoder_params(para, x.shape[-1], IMS, lid, NLAYER)
        hs = x.shape[-1]
        p["attn_qkvb"][hs + 5], p["attn_qkvb"][2 * hs + 6] = INF, -INF
        p["encdec_attn_qw"][3, 4], p["encdec_attn_ow"][7, 8] = INF, -INF
        p["output_w"][1, 3] = INF
        if lid == 0:
            p["encdec_attn_kvw"][9, 10] = -INF
    layers = _make_stack(paras, True, "relu", 64, 32)
    try:
        with np.errstate(all="ignore"):
            kv = lo.decoder_encdec_kv(paras[0], enc, NH, IMS, NLAYER)
        for lid, layer in enumerate(layers):
            with np.errstate(all="ignore"):
                want = lo.decoder_layer_forward(paras[lid], lid, NLAYER, x, kv, mask, NH, IMS, True, "relu")
            with torch.no_grad():
                got = layer(to_dev(x), to_dev(enc).transpose(0, 1), to_dev(pad))
            _check(got, want, np.ones(x.shape[:2], bool))
    finally:
        _release(layers)


@pytest.mark.parametrize("hs,nh,pre_ln", [(1536, 24, False), (2080, 65, True), (4096, 32, False), (4128, 129, False),
                                          (4128, 129, True), (5120, 40, True)])
def test_wide_layers(hs, nh, pre_ln):
    """The layer norm by every number of registers a row takes, and by rereading it beyond 4096."""
    from test_oracle_layer_ops import config0
    batch, seq, ims = 2, 5, 64
    cfg0 = config0(np.random.default_rng(hs), pre_ln, "gelu", batch, seq, hs, nh, ims)
    layer, para = _make_layer(cfg0, pre_ln, "gelu", nh, 16, 8)
    x = cfg0[1].astype(np.float16)
    with torch.no_grad():
        got = layer(to_dev(x), torch.zeros(batch, seq, device="cuda"))
    want = _lo().encoder_layer_forward(para, x, np.zeros((batch, seq), np.float16), nh, ims, pre_ln, "gelu")
    # a code of the output projection that another order of sums moves by one is one step of it,
    # which grows with the width
    _check(got, want, np.ones((batch, seq), bool), 2e-2 + cfg0[2]["out_out"] / 127)


def test_encoder_output_at_any_place():
    """A view that is not 16-byte aligned, or whose strides are no multiples of 8, gives the bits of
    an aligned tensor (a stride that a single sentence or token does not use says nothing);
    the C call refuses what its contract excludes."""
    from lightseq_amd import lib
    for batch, src in ((2, 12), (1, 12), (2, 1)):
        paras, x, enc, pad, mask = _case(7, batch, 9, src)
        layers = _make_stack(paras, True, "relu", 64, 32)
        layer, hs = layers[0], x.shape[-1]
        try:
            xd, padd = to_dev(x), to_dev(pad)
            aligned = to_dev(np.ascontiguousarray(enc.transpose(1, 0, 2)))
            n = aligned.numel()
            odd = torch.empty(n + 8, dtype=torch.half, device="cuda")[3:n + 3].view(aligned.shape).copy_(aligned)
            assert odd.is_contiguous() and odd.data_ptr() % 16 == 6
            wide = torch.empty(src, batch, hs + 4, dtype=torch.half, device="cuda")[..., :hs].copy_(aligned)
            places = [odd, wide]
            if batch == 1:
                places.append(aligned.as_strided(aligned.shape, (hs, 7, 1)))
            if src == 1:
                places.append(aligned.as_strided(aligned.shape, (7, hs, 1)))
            with torch.no_grad():
                want = layer(xd, aligned, padd)
                for place in places:
                    assert torch.equal(layer(xd, place, padd), want)
            out = torch.empty_like(xd)

            def call(address, stride_b, stride_s):
                lib.call("ls_decoder_layer_call_fp16", 0, lib.ptr(layer.para), lib.ptr(xd), address, stride_b,
                         stride_s, lib.ptr(padd), 1, lib.ptr(out), batch, 9, src, -1, *[None] * 5, 0, 1,
                         lib.current_stream())

            refused = [(odd.data_ptr(), hs, batch * hs)]
            if batch > 1:
                refused.append((aligned.data_ptr(), 4, batch * hs))
            if src > 1:
                refused.append((aligned.data_ptr(), hs, 4))
            for args in refused:
                with pytest.raises(lib.LSHError, match="16-byte aligned"):
                    call(*args)
            call(aligned.data_ptr(), hs, batch * hs)
            assert torch.equal(out, want)
        finally:
            _release(layers)
