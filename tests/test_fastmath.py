"""The transport's in-range elementary functions, divisions and roots and its generator steps (fastmath.h,
ranecu.h) have the bits of the general ones, which the oracle shares, over their stated ranges: on every
float or state where the range is a set of those, on drawn arguments otherwise."""
import numpy as np
import pytest

import mcpet


def _bits(x):
    return int(np.float32(x).view(np.uint32))


INF = _bits(np.inf)
# how many floats (of 2^32 bit patterns) or states (of 2^31) each range holds
IN_RANGE = {"floor": 2 * (INF + 1), "floor_nan": 2 ** 32, "sqrtf": 2 + INF - _bits(2.0 ** -100) - 1,
            "logf": INF - _bits(2.0 ** -126), "expf": 2 ** 32 - (INF - _bits(88.0)), "sincosf": 2 * _bits(8192.0),
            "div_1000": INF + 1 + INF - _bits(2.0 ** -80), "ranecu": 2147483562}
DRAWN = ("divf", "divf_r", "div", "sqrt", "log", "exp", "sincos")


@pytest.mark.gpu
@pytest.mark.parametrize("name", mcpet.FAST_FUNCTIONS)
def test_in_range_functions_equal_the_general_ones(name):
    first, n = (0, 2 ** (31 if name == "ranecu" else 32)) if name in IN_RANGE else (2026, 2 ** 31)
    print(name, n, flush=True)
    differ, at, compared = mcpet.selftest_fastmath(name, first, n)
    assert differ == 0, f"{name}: {differ} of {compared} differ, the first at {first + at:#x}"
    assert compared == IN_RANGE[name] if name in IN_RANGE else compared > n // 2


def test_the_self_test_rejects_bad_arguments_without_a_device():
    assert sorted(list(IN_RANGE) + list(DRAWN)) == sorted(mcpet.FAST_FUNCTIONS)
    assert mcpet.lib().mcpet_selftest_fastmath(0, 0, 0, None) == 1
