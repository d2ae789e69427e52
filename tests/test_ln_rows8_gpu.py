"""Layer norms of 8-wide rows at the edges of their lane layouts: rows that fill the lanes' chunks
exactly and rows one chunk short of or beyond that, one row and an odd number of them."""
import numpy as np
import pytest

import test_kernels_gpu as tk

pytestmark = pytest.mark.gpu

SHAPES = [(rows, hidden) for rows in (1, 3) for hidden in (8, 248, 256, 264, 504, 760, 1016, 1032, 1536, 2040)]


@pytest.mark.parametrize("dtype", tk.DTYPES)
@pytest.mark.parametrize("acc_dtype", [np.int8, np.int32])
@pytest.mark.parametrize("shape", SHAPES)
def test_residual_bias_ln_i8O(oracle, rng, dtype, acc_dtype, shape):
    tk.test_residual_bias_ln_i8O(oracle, rng, dtype, acc_dtype, shape[0] == 3, shape[1] % 16 == 0, shape)


@pytest.mark.parametrize("dtype", tk.DTYPES)
@pytest.mark.parametrize("shape", SHAPES)
def test_first_and_last_norm(oracle, rng, dtype, shape):
    tk.test_norm_layer_resual_i8O(oracle, rng, dtype, shape[0] == 3, shape)
    tk.test_residual_bias_ln_i32I(oracle, rng, dtype, shape[1] % 16 == 0, shape)
