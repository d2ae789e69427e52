"""The layers' quantiser divides by a reciprocal and one residual correction (layer_device.h): the codes
of every half are those of the division, for both quantisers."""
import numpy as np
import pytest

HALFS = np.arange(65536, dtype=np.uint16).view(np.float16)
HALFS = HALFS[~np.isnan(HALFS)].astype(np.float32)


def _fma(a, b, c):
    """Rounded once: the product is exact in extended precision."""
    return (a.astype(np.longdouble) * np.longdouble(b) + c).astype(np.float32)


@pytest.mark.parametrize("signed", [True, False])
def test_codes_are_those_of_the_division(signed):
    f32 = np.float32
    rng = np.random.default_rng(3)
    clips = np.concatenate([[1, 2, 0x03ff, 0x0400, 0x3c00, 0x57f0, 0x7bff],
                            rng.integers(1, 0x7c00, size=160)]).astype(np.uint16).view(np.float16).astype(f32)
    with np.errstate(all="ignore"):
        for c in clips:
            scale = c / f32(127) if signed else c / f32(127) / f32(2)
            shift = f32(0) if signed else f32(127)
            want = np.clip(np.floor((HALFS / scale - shift) + f32(0.5)), -127, 127)
            inv = f32(1) / scale
            x = np.clip(HALFS, -c if signed else f32(0), c)
            q = (x * inv).astype(f32)
            q = _fma(_fma(q, -scale, x), inv, q)
            np.testing.assert_array_equal(np.floor((q - shift) + f32(0.5)), want, err_msg=str(c))
