"""Blocked operands of 4 GiB and more: the rows behind the 2^32nd byte."""
import pytest
import torch

from helpers import DEV
from test_layer_ops_gpu import _make_layer

pytestmark = pytest.mark.gpu


# whole 128-byte steps of K (the LDS tiles), an odd number of 64-byte slices (the split of K), and
# weights instead of activations
@pytest.mark.parametrize("m,n,k", [(65568, 64, 65536), (65568, 64, 65600), (16, 65600, 65536)])
def test_int8_product(m, n, k):
    from lightseq_amd import kernels as K
    g = torch.Generator(device=DEV).manual_seed(k)
    a, w = (torch.randint(-127, 128, (rows, k), dtype=torch.int8, device=DEV, generator=g) for rows in (m, n))
    assert max(m, n) * k >= 2 ** 32
    ab, wb = K.block_rows(a), K.block_rows(w)
    c = torch.zeros(m, n, dtype=torch.int32, device=DEV)
    K.gemm_i8_blocked_i32o(ab, wb, c, m, n, k)
    for rows in (slice(0, 48), slice(m - 48 if m > 48 else 0, m)):
        for cols in (slice(0, 64), slice(n - 64, n)):
            want = a[rows].double() @ w[cols].double().t()
            assert torch.equal(c[rows, cols].double(), want)


def test_encoder_layer():
    """524800 tokens with an inner size of 4096: the fp16 activation between the feed-forward
    products has 4.3 GB.  Sequences on both sides of the 2^32nd byte have the bits of a small batch."""
    import numpy as np
    from test_oracle_layer_ops import config0
    seq, batch = 64, 8200
    cfg0 = config0(np.random.default_rng(3), False, "relu", 2, seq, 64, 1, 4096)
    layer, _ = _make_layer(cfg0, False, "relu", 1, batch * seq, seq)
    assert batch * seq * 4096 * 2 >= 2 ** 32
    g = torch.Generator(device=DEV).manual_seed(0)
    x = torch.randn(batch, seq, 64, device=DEV, generator=g).half()
    pad = torch.zeros(batch, seq, device=DEV)
    with torch.no_grad():
        full = layer(x, pad)
        for part in (slice(0, 8), slice(8188, 8200)):
            assert torch.equal(layer(x[part].contiguous(), pad[part].contiguous()), full[part])
