"""The wave step on directional fields whose neighbouring values lie far apart:
a second-order upwind value 1.5 a - 0.5 b with b many orders below a, where
forming it in double and rounding that to float is not one rounding of the
exact value, and bins in the subnormal range.  Bit for bit the oracle's."""
import numpy as np
import pytest
from test_gpu_wave_tiles import CASES, FIELDS, build, oracle_step

pytestmark = pytest.mark.gpu


def spread(rng, shape, low):
    """Values of 24 random bits, each down by none or low .. low + 8 powers of two."""
    m = rng.integers(1 << 23, 1 << 24, shape).astype(np.float64) * 2.0 ** -23
    return np.ldexp(m, -np.where(rng.random(shape) < 0.5, 0, rng.integers(low, low + 9, shape)))


@pytest.mark.parametrize("n", [1, 2, 7, 9, 10, 14, 16])
@pytest.mark.parametrize("where", ["apart", "subnormal"])
def test_far_apart_neighbours(need_gpu, n, where):
    d, o, S, Q, Trep = build(n, *CASES[n][:3], CASES[n][3])
    rng = np.random.default_rng(90 + n)
    for f in ("ee", "rr"):
        shape = d.get(f).shape
        if where == "apart":
            a = 50.0 * spread(rng, shape, 46)
        else:  # 2^-149 .. 2^-120
            a = np.ldexp(spread(rng, shape, 8), -rng.integers(126, 141, shape))
        a = a.astype(np.float32)
        d.set(f, a)
        o.set(f, a)
    t0, dt = 150.0, 0.3
    for k in range(2):
        t = t0 + (k + 1) * dt
        d.use_bnd_record(0, t - t0, 1.0, Trep)
        d.step(dt, t)
        oracle_step(o, S, Q, Trep, t0, t, dt)
        for f in FIELDS:
            assert np.array_equal(d.get(f), o.get(f), equal_nan=True), (k, f)
    d.close()
