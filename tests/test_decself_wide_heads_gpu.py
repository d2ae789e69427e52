"""Decoder self attention over caches that one wavefront's loads cover: every dimension of a head is
written, also where a head has more of them than a wavefront has lanes."""
import numpy as np
import pytest
import torch

from conftest import assert_codes_close
from helpers import DEV, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("step_num", [1, 31, 33, 63, 64])
def test_short_caches(oracle, rng, d, step_num):
    from lightseq_amd import kernels as K
    rows, heads, max_step = 5, 3, 70
    q, kc, vc = (rng.integers(-127, 128, size=s, dtype=np.int8)
                 for s in ((rows, heads * d), (rows, heads, max_step, d), (rows, heads, max_step, d)))
    dq, qs, scale = 0.5 / 127, 127 / 1.5, float(np.float16(np.sqrt(1.0 / d)))
    want = oracle.fuse_softmax_new_value_i32I_i8O(oracle.decself_scores(q, kc, step_num), vc, step_num, scale, dq, qs)
    out = torch.full((rows, heads * d), 99, dtype=torch.int8, device=DEV)
    K.decself_attention_i8(to_dev(q), to_dev(kc), to_dev(vc), out, rows * heads, step_num, max_step, heads, d, scale,
                           dq, qs)
    assert_codes_close(to_np(out), want, what="decself_attention")
