"""sinh and tanh are odd, zeros and infinities included, as in C99 Annex F."""
import math

import numpy as np
import pytest
from test_xmath import xm


@pytest.mark.parametrize("name", ["sinh", "tanh"])
@pytest.mark.parametrize("is_float", [False, True])
def test_odd_functions(name, is_float):
    x = np.array([0.0, 5e-324, 1e-300, 1e-45, 1e-38, 1e-8, 0.5, 1.0, 21.9, 22.1, 88.0, 700.5, 1e4, math.inf])
    if is_float:
        x = x.astype(np.float32).astype(np.float64)
    a, b = xm(name, x, is_float=is_float), xm(name, -x, is_float=is_float)
    assert np.array_equal(np.signbit(b), np.ones(len(x), bool)) and not np.signbit(a).any()
    assert np.array_equal(a, -b)
    assert a[0] == 0.0 and a[-1] == (math.inf if name == "sinh" else 1.0)
    assert math.isnan(xm(name, [math.nan], is_float=is_float)[0])
