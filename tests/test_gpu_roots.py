"""The device's reciprocal and square root, which take a short form where it is
correctly rounded, against IEEE arithmetic (numpy's binary32), bit for bit:
every significand at exponents of both parities over the range, at its ends
and around the root's lower end of the short form (2^-96), both signs, and
zeros, infinities, NaN and the smallest and largest numbers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPECIAL = np.array([0x00000000, 0x80000000, 0x00000001, 0x80000001, 0x007fffff, 0x00800000, 0x00800001, 0x7f7fffff,
                    0xff7fffff, 0x7f800000, 0xff800000, 0x7fc00000, 0x7e800000, 0x7e7fffff, 0x7e800001, 0x0f800000,
                    0x0f7fffff, 0x0f800001], np.uint32).view(np.float32)


def same(got, want):
    return ((got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))).all()


@pytest.mark.parametrize("exponent", [0, 1, 2, 30, 31, 32, 63, 126, 127, 128, 200, 252, 253, 254])
def test_rcp_and_sqrt_every_significand(ctx, exponent):
    x = ((np.uint32(exponent) << np.uint32(23)) | np.arange(1 << 23, dtype=np.uint32)).view(np.float32)
    with np.errstate(all="ignore"):
        assert same(ctx.math_eval("rcp", x), np.float32(1.0) / x)
        assert same(ctx.math_eval("rcp", -x), np.float32(1.0) / -x)
        assert same(ctx.math_eval("sqrt", x), np.sqrt(x))


def test_rcp_and_sqrt_special(ctx):
    with np.errstate(all="ignore"):
        assert same(ctx.math_eval("rcp", SPECIAL), np.float32(1.0) / SPECIAL)
        assert same(ctx.math_eval("sqrt", SPECIAL), np.sqrt(SPECIAL))
