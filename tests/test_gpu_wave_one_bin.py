"""A single direction bin has no directional advection, whatever its width: a
run without directional spread has one bin of width 0 (thetamin = thetamax).
A step equals the oracle's bit for bit."""
import numpy as np
import pytest
from test_gpu_wave_tiles import FIELDS, oracle_step

from oracle.pyorc import Oracle
from xbeach_gpu_amd import Domain, setups

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{}, dict(wci=1.0, hwci=0.5), dict(roller=0)], ids=["plain", "currents", "no roller"])
@pytest.mark.parametrize("dtheta", [0.0, 120.0, 60.0])
def test_one_bin(need_gpu, dtheta, kw):
    nx, ny = 70, 19
    p = setups.small_params(nx=nx, ny=ny, dtheta=120.0, **kw)
    assert p.ntheta == 1
    st = setups.spun_up_state(p, setups.small_bathy(nx, ny, p.dx), seed=61)
    rng = np.random.default_rng(3)
    S = rng.uniform(0.0, 400.0, (3, ny, 1)).astype(np.float32)
    Q = rng.uniform(-0.1, 0.1, (3, 4, ny)).astype(np.float32)
    p.dtheta = dtheta * np.pi / 180.0
    d, o = Domain(p), Oracle(p, 4)
    for k, v in st.items():
        d.set(k, v)
        o.set(k, v)
    d.init_state(9.0)
    o.init_state(9.0)
    d.set_bnd_series(S, Q)
    t0, dt = 150.0, 0.1
    d.use_bnd_record(0, dt, 1.0, 9.0)
    d.step(dt, t0 + dt)
    oracle_step(o, S, Q, 9.0, t0, t0 + dt, dt)
    assert np.isfinite(o.get("ee")).all()
    for f in FIELDS:
        assert np.array_equal(d.get(f), o.get(f), equal_nan=True), f
    d.close()
