"""Attention over more than 128 keys at the edges of its blocks: of 32 and 128 keys, of the 32-query
tiles, sequences of a packed batch that end anywhere, blocks that are masked in part and as a whole."""
import numpy as np
import pytest
import torch

from helpers import DEV, to_dev, to_np

pytestmark = pytest.mark.gpu


def _reference(q, k, v, mask, causal):
    """float64 over fp16 operands, rounded where the kernels round: scores, probabilities, context."""
    s = (np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k.astype(np.float64)) * 0.125).astype(np.float16)
    s = s.astype(np.float64)
    if mask is not None:
        s = s + mask.astype(np.float64)[:, None, None, :]
    if causal:
        n = s.shape[-1]
        s = np.where(np.arange(n)[None, :] > np.arange(s.shape[2])[:, None], -np.inf, s)
    m = s.max(-1, keepdims=True)
    e = np.exp(s - np.where(np.isfinite(m), m, 0))
    t = e.sum(-1, keepdims=True)
    p = np.where(t > 0, e / np.where(t > 0, t, 1), 0).astype(np.float16)
    return np.einsum("bhqk,bhkd->bhqd", p.astype(np.float64), v.astype(np.float64))


@pytest.mark.parametrize("batch,heads,q_len,k_len,causal", [
    (2, 2, 129, 129, False), (1, 3, 160, 160, True), (1, 1, 256, 256, True), (2, 1, 257, 257, False),
    (1, 2, 384, 384, True), (40, 4, 385, 385, False), (1, 1, 512, 512, False), (1, 1, 513, 513, False),
    (2, 2, 1, 200, False), (3, 1, 33, 300, False),
])
def test_layer_attention(batch, heads, q_len, k_len, causal):
    from test_decoder_layer_gpu import _ops
    rng = np.random.default_rng(k_len)
    q, k, v = ((rng.standard_normal((batch, heads, n, 64)) * 1.5).astype(np.float16) for n in (q_len, k_len, k_len))
    mask = np.zeros((batch, k_len), np.float16)
    with np.errstate(over="ignore"):
        for b in range(batch):
            mask[b, k_len - (b * 37) % 70:] = np.float16(-1e8) if b else 0  # the first one has no padding
    mask[-1, 5] = -2.5        # any addend counts
    mask[-1, 64:96] = -np.inf  # a block of 32 masked as a whole
    got = torch.zeros(batch, q_len, heads * 64, dtype=torch.float16, device=DEV)
    _ops().layer_cross_attention(to_dev(q), to_dev(k), to_dev(v), to_dev(mask), got, batch, q_len, k_len, heads, 64,
                                 causal)
    want = _reference(q, k, v, mask, causal).transpose(0, 2, 1, 3).reshape(batch, q_len, heads * 64)
    np.testing.assert_allclose(to_np(got).astype(np.float64), want, atol=8e-3)  # (a score around 16 is rounded to 1 / 64)
