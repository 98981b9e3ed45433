"""The FP32 reciprocal of the adjoint's pair bodies (rcp_n in sph_device.h): one
Newton step on the hardware's approximation y, y + y (1 - x y) with fused
multiply-adds.  For every mantissa of x and every y within an ulp of 1/x (the
hardware's bound; 0.882 measured) the result is within 0.500001 ulp: 1 - x y is
exact before its rounding and at most 2^-22, so what remains is the last
rounding, (2^-22)^2 and 2^-22 2^-24."""
import numpy as np


def newton(x, y):
    """fma(fma(-x, y, 1), y, y): the products of two floats are exact in FP64,
    and so is 1 - x y; the last sum's FP64 rounding is 2^-29 of an ulp."""
    e = (1.0 - x.astype(np.float64) * y).astype(np.float32)
    return (e.astype(np.float64) * y + y).astype(np.float32)


def test_newton_step_rounds_as_a_division():
    for lo in range(0, 1 << 23, 1 << 20):
        x = (1.0 + np.arange(lo, lo + (1 << 20)) * 2.0 ** -23).astype(np.float32)
        t = 1.0 / x.astype(np.float64)
        near = t.astype(np.float32)
        ulp = np.spacing(np.minimum(near, np.float32(1.0) - np.float32(2.0 ** -24)))
        for y in (near, np.nextafter(near, np.float32(0)), np.nextafter(near, np.float32(2))):
            ok = np.abs(y - t) <= ulp
            err = np.abs(newton(x, y) - t)[ok] / ulp[ok]
            assert err.max() <= 0.500001, (lo, err.max())
