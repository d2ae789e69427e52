"""Products on blocked operands against exact integer products and the row-major kernels, at the
edges of the tiles, of the K ranges and of the dispatch between the two kernels."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (m, n, k): one row; partial 16-row blocks and column tiles; K of 1, 2, 3, 12, 16 slices of 64 bytes;
# every tile of the small kernel; several rounds of the chip; the LDS tile kernel with remainders
SHAPES = [(1, 64, 64), (16, 256, 128), (17, 100, 192), (5, 2304, 768), (33, 1024, 1024), (64, 4096, 1024),
          (65, 768, 3072), (130, 3072, 768), (330, 768, 768), (530, 1152, 512), (1000, 1024, 4096),
          (2561, 768, 768), (2561, 3072, 768), (4100, 2304, 768), (1024, 50272, 128)]


def _codes(rng, rows, k):
    return rng.integers(-127, 128, size=(rows, k), dtype=np.int8)


def _product(a, w):
    return (torch.from_numpy(a).to(DEV).double() @ torch.from_numpy(w).to(DEV).double().t()).to(torch.int32)


@pytest.mark.parametrize("rows,k", [(1, 64), (15, 128), (16, 64), (35, 768)])
def test_block_rows_layout_and_back(rng, rows, k):
    from lightseq_amd import kernels as K
    x = _codes(rng, rows, k)
    b = K.block_rows(torch.from_numpy(x).to(DEV))
    want = np.zeros(((rows + 15) // 16 * 16, k), np.int8)
    want[:rows] = x
    want = want.reshape(-1, 16, k // 64, 4, 16).transpose(0, 2, 3, 1, 4).reshape(-1)
    np.testing.assert_array_equal(b.cpu().numpy(), want)
    np.testing.assert_array_equal(K.block_rows(b, (rows, k, torch.int8)).cpu().numpy(), x)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_int32_and_requantised_outputs(rng, m, n, k):
    from lightseq_amd import kernels as K
    a, w = _codes(rng, m, k), _codes(rng, n, k)
    ab, wb = K.block_rows(torch.from_numpy(a).to(DEV)), K.block_rows(torch.from_numpy(w).to(DEV))
    want = _product(a, w)
    c = torch.full((m, n), -7, dtype=torch.int32, device=DEV)
    K.gemm_i8_blocked_i32o(ab, wb, c, m, n, k)
    assert torch.equal(c, want)
    alpha = float(np.float32(0.3 / (127 * k ** 0.5)))
    c8 = torch.zeros(m, n, dtype=torch.int8, device=DEV)
    K.gemm_i8_blocked_i8o(ab, wb, c8, m, n, k, alpha)
    q = torch.floor(want.to(torch.float32) * alpha + 0.5).clamp(-127, 127).to(torch.int8)
    assert torch.equal(c8, q)


@pytest.mark.parametrize("m,n,k,ks", [(16, 1024, 4096, 4), (40, 768, 3072, 2), (3, 64, 256, 4)])
def test_split_k_planes(rng, m, n, k, ks):
    from lightseq_amd import kernels as K
    a, w = _codes(rng, m, k), _codes(rng, n, k)
    c = torch.zeros(ks, m, n, dtype=torch.int32, device=DEV)
    K.gemm_i8_blocked_i32o(K.block_rows(torch.from_numpy(a).to(DEV)), K.block_rows(torch.from_numpy(w).to(DEV)),
                           c, m, n, k, ks)
    assert torch.equal(c.sum(0).to(torch.int32), _product(a, w))


@pytest.mark.parametrize("m,n,k", [s for s in SHAPES if s[1] % 64 == 0 and s[1] <= 4096])
def test_table_epilogue(rng, m, n, k):
    from lightseq_amd import kernels as K
    a, w = _codes(rng, m, k), _codes(rng, n, k)
    lut = torch.from_numpy(rng.integers(-127, 128, size=(n, 256), dtype=np.int8)).to(DEV)
    alpha = float(np.float32(0.3 / (127 * k ** 0.5)))
    out = torch.zeros((m + 15) // 16 * 16 * n, dtype=torch.int8, device=DEV)
    K.gemm_i8_blocked_lut_i8o(K.block_rows(torch.from_numpy(a).to(DEV)), K.block_rows(torch.from_numpy(w).to(DEV)),
                              out, lut, m, n, k, alpha)
    q = torch.floor(_product(a, w).to(torch.float32) * alpha + 0.5).clamp(-127, 127).to(torch.int64)
    want = torch.gather(lut.t(), 0, q + 128)  # lut[n][code + 128]
    assert torch.equal(K.block_rows(out, (m, n, torch.int8)), want)


@pytest.mark.parametrize("rows,heads,d,beam", [(1, 4, 64, 1), (16, 16, 64, 4), (20, 12, 32, 4), (64, 16, 64, 4)])
def test_generation_epilogues_leave_the_row_major_bytes(rng, rows, heads, d, beam):
    from lightseq_amd import kernels as K
    H, steps, at = heads * d, 9, 5
    a, w, wq = _codes(rng, rows, H), _codes(rng, 3 * H, H), _codes(rng, H, H)
    bias = (torch.from_numpy(rng.standard_normal(3 * H).astype(np.float32)) * 0.2).half().to(DEV)
    da, dw, dwq = (torch.from_numpy(t).to(DEV) for t in (a, w, wq))
    alpha, dq, qs = float(np.float32(0.3 / (127 * H ** 0.5))), 0.031, 21.0
    outs = []
    for blocked in (False, True):
        q = torch.zeros(rows, H, dtype=torch.int8, device=DEV)
        kc, vc = (torch.zeros(rows, heads, steps, d, dtype=torch.int8, device=DEV) for _ in range(2))
        f = K.gemm_i8_blocked_decself_qkv_i8o if blocked else K.gemm_i8_decself_qkv_i8o
        f(K.block_rows(da) if blocked else da, K.block_rows(dw) if blocked else dw, bias, q, kc, vc, rows, H, H,
          heads, steps, at, alpha, dq, qs)
        outs.append([q, kc, vc])
        if rows % beam == 0:
            eq = torch.zeros(rows, H, dtype=torch.half, device=DEV)
            g = K.gemm_i8_blocked_encdec_q if blocked else K.gemm_i8_encdec_q
            g(K.block_rows(da) if blocked else da, K.block_rows(dwq) if blocked else dwq, bias, eq, rows, H, H, beam,
              heads, alpha, dq)
            outs[-1].append(eq)
    for x, y in zip(*outs):
        assert torch.equal(x, y)
