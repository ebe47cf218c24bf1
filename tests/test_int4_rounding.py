"""The division-free code and scale arithmetic of the int4 pack kernels, step by step in numpy (float64
holds every product and sum before its one rounding to float32), against the IEEE division, rint and
clamp that define them -- over every pair of 11-bit significands at the exponents where they meet."""

import numpy as np
import pytest

F = np.float32


def codes(x, rs):
    t = (x.astype(np.float64) * rs.astype(np.float64) + 384.0).astype(F)      # fma, one rounding
    t = t + F(12582912.0 - 384.0)
    return np.clip(t, F(12582904), F(12582919)).astype(np.float64) - 12582912.0


@pytest.mark.parametrize("ulp", [-1, 0, 1])   # v_rcp_f32 is within one ulp of 1 / s
@pytest.mark.parametrize("shift", range(-3, 5))
def test_codes_equal_rounded_division(shift, ulp):
    x = (np.arange(1024, 2048, dtype=np.float64) * 2.0 ** shift).astype(F)[None, :]
    for part in np.array_split(np.arange(1024, 2048), 8):
        s = part.astype(F)[:, None]
        rs = (F(1) / s).astype(F)
        rs = np.nextafter(rs, F(np.inf) * ulp if ulp else rs, dtype=F)
        want = np.clip(np.rint((x / s).astype(F)), -8, 7)
        assert np.array_equal(codes(x, rs), want)
        assert np.array_equal(codes(-x, rs), np.clip(np.rint((-x / s).astype(F)), -8, 7))


def test_codes_of_extreme_quotients():
    x = np.array([3.4e38, -3.4e38, np.inf, -np.inf, 0.0, -0.0, 1e-30], dtype=F)
    rs = np.full_like(x, F(1) / F(65504))
    with np.errstate(invalid="ignore", over="ignore"):
        assert codes(x, rs).tolist() == [7, -8, 7, -8, 0, 0, 0]


def test_group_scale_equals_divided_scale():
    """fp16(fp32(a / 7)) for every 11-bit significand at every exponent from fp16's subnormals to
    past its range."""
    a = (np.arange(1024, 2048, dtype=np.float64)[None, :] * 2.0 ** np.arange(-40, 40)[:, None]).astype(F).ravel()
    q = (a * (F(1) / F(7))).astype(F)
    e = (a.astype(np.float64) - 7.0 * q.astype(np.float64)).astype(F)
    got = (e.astype(np.float64) * np.float64(F(1) / F(7)) + q.astype(np.float64)).astype(F)
    with np.errstate(over="ignore"):
        assert np.array_equal(got.astype(np.float16), (a / F(7)).astype(F).astype(np.float16))
