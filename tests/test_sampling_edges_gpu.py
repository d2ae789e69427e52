"""Random sampling where the reading of a row can go wrong: fewer ids than classes, parts of 16-byte
pieces at either end (rows at every alignment), one pass of the registers (65536 ids) and more, rows of
one code, the lowest code.  Against the oracle; a draw within 1e-5 of a boundary of the cumulative
distribution (another order of float sums) is compared by membership only."""
import numpy as np
import pytest
import torch

from helpers import DEV, to_np
from oracle import sampling as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 15, 300, 1023, 1025, 4097, 16385, 65521, 65536, 65537, 70001, 131073])
@pytest.mark.parametrize("k,p", [(2, 0.0), (32, 0.0), (0, 0.9)])
def test_rows_of_every_alignment(vocab, k, p):
    from lightseq_amd import kernels as kk
    rng = np.random.default_rng(vocab + k)
    batch, scale, seed = 5, 0.07, 11
    logits = np.clip(rng.normal(0, 28, size=(batch, vocab)), -128, 127).astype(np.int8)
    logits[1] = -128  # (every id ties)
    logits[2] = 5
    state = kk.rng_setup(batch, seed)
    ids = torch.zeros(batch, 4, dtype=torch.int32, device=DEV)
    last = torch.zeros(batch, dtype=torch.int32, device=DEV)
    unf = torch.zeros(1, dtype=torch.int32, device=DEV)
    flat = torch.full((batch * vocab + 16,), 127, dtype=torch.int8, device=DEV)  # what is not the row's would win
    at = vocab % 13
    flat[at:at + batch * vocab] = torch.from_numpy(logits.reshape(-1)).to(DEV)
    kk.gpt_sample_step(flat[at:], ids, last, vocab, 4, 1, batch, unf, vocab + 1, k, p, scale, state)
    got = to_np(last)
    for b in range(batch):
        u = S.uniform_of_draw(seed, b, 0)
        tok, amb, cand, _ = S.topk_sample_row(logits[b], k, scale, u) if k else S.topp_sample_row(logits[b], p, scale, u)
        if not amb:
            assert got[b] == tok, b
        elif k:
            assert got[b] in cand, b
        else:
            assert 0 <= got[b] < vocab
