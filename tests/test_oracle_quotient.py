"""The quotient of the iteration kernels (p2_quotient in poker2_amd/csrc/common.h), restated in C with fused multiply-adds
(oracle/quotient.c), against IEEE division for every mantissa of the divisor."""
import ctypes

import pytest

from oracle import ranker_c


def differs(eb: int, ea: int, wide: bool = False, step: int = 1, dividends: int = 6) -> tuple[int, int]:
    f = ranker_c.lib().p2o_quotient_differs
    f.restype = ctypes.c_int64
    f.argtypes = [ctypes.c_int] * 3 + [ctypes.c_int64, ctypes.c_int, ctypes.c_void_p]
    worst = ctypes.c_int64()
    return f(eb, ea, int(wide), step, dividends, ctypes.byref(worst)), worst.value


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("eb,ea", [(0, 0), (-27, -27), (-27, -28), (0, -102), (-27, -102), (100, 100), (125, 125), (125, 24),
                                   (126, 126), (-27, 99)])
def test_equal_to_division(eb, ea, wide):
    """Exponents of divisor and dividend: sums and masses from the kernels' thresholds (1e-8 = 2^-27) up to the largest a
    reciprocal is a normal number for, dividends down to 2^-102."""
    assert differs(eb, ea, wide) == (0, 0)


def test_divisors_below_those_of_the_wide_reciprocal():
    assert differs(-126, -102) == (0, 0) and differs(-126, -100) == (0, 0)
    assert differs(-94, -94, wide=True) == (0, 0)


@pytest.mark.parametrize("eb,ea", [(0, -110), (0, -126), (-27, -126),       # the remainder is rounded to a multiple of 2^-149
                                   (115, -20), (60, -80), (127, 127)])       # a subnormal quotient, or reciprocal
def test_a_unit_in_the_last_place_elsewhere(eb, ea):
    assert differs(eb, ea, step=5)[1] <= 1
    assert differs(eb, ea, wide=True, step=5)[1] <= 1


def test_an_overflowing_quotient_is_not_infinity():
    """What the comment beside the quotient says the kernels' divisors keep away."""
    assert differs(-27, 101, step=1 << 12)[0] > 0
