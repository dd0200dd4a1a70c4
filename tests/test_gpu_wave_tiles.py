"""Every instantiation of the wave kernel (bin classes, counts known to the
compiler or not, currents, roller off, representative periods and direction
steps beyond the reciprocals' range) over the tile layouts its rows can meet:
one row or all rows of the last tile inside the domain, rows 0 and ny-1 within
one tile height, a ragged last column tile.  Two steps equal the CPU oracle's
bit for bit, both sides performing the same operations in the same order."""
import numpy as np
import pytest

from oracle.pyorc import Oracle
from xbeach_gpu_amd import Domain, setups
from xbeach_gpu_amd.ensemble import Ensemble, RunSetup

pytestmark = pytest.mark.gpu

FIELDS = ("ee", "rr", "H", "E", "R", "DR", "D", "urms", "ust", "thetamean", "Sxx", "Syy", "Sxy", "Fx", "Fy", "zs", "uu",
          "vv", "C", "zb")
# bins, nx, ny, options
CASES = [
    (1, 70, 19, {}),                       # dtheta of 2.09 rad
    (5, 130, 9, {}),
    (9, 64, 17, dict(wci=1.0, hwci=0.5)),
    (12, 65, 8, {}),
    (12, 128, 25, dict(wci=1.0, hwci=0.5)),
    (12, 63, 4, dict(roller=0)),
    (13, 40, 10, {}),
    (18, 66, 33, dict(roller=0)),
    (18, 129, 7, dict(wci=1.0, hwci=0.5)),
    (24, 64, 9, {}),
    (24, 100, 16, dict(wci=1.0, hwci=0.5)),
    (24, 33, 41, dict(roller=0, wci=1.0, hwci=0.5)),
    (24, 48, 12, dict(Trep=2.5)),          # sigm above 2
    (25, 67, 17, {}),
    (36, 64, 6, dict(wci=1.0, hwci=0.5)),
    (40, 31, 9, {}),
    (64, 65, 18, dict(wci=1.0, hwci=0.5)),
    (64, 20, 5, dict(roller=0)),
]


def build(n, nt, nx, ny, kw):
    kw = dict(kw)
    Trep = kw.pop("Trep", 9.0)
    p = setups.small_params(nx=nx, ny=ny, dtheta=120.0 / nt, **kw)
    assert p.ntheta == nt
    st = setups.spun_up_state(p, setups.small_bathy(nx, ny, p.dx), seed=50 + n)
    rng = np.random.default_rng(n)
    S = rng.uniform(0.0, 400.0, (3, ny, nt)).astype(np.float32)
    Q = rng.uniform(-0.1, 0.1, (3, 4, ny)).astype(np.float32)
    d, o = Domain(p), Oracle(p, 4)
    for k, v in st.items():
        d.set(k, v)
        o.set(k, v)
    d.init_state(Trep)
    o.init_state(Trep)
    d.set_bnd_series(S, Q)
    return d, o, S, Q, Trep


def oracle_step(o, S, Q, Trep, t0, t, dt):
    rec = int(np.floor(t - t0))
    tsl = t - (t0 + rec)
    St = (S[rec].astype(np.float64) + tsl * (S[rec + 1].astype(np.float64) - S[rec])).astype(np.float32)
    o.set_forcing(St, Q[rec], Q[rec + 1], Trep, tsl, 1.0)
    o.step(dt, t)


@pytest.mark.parametrize("n", range(len(CASES)), ids=lambda n: "{}x{}x{}-{}".format(
    CASES[n][1], CASES[n][2], CASES[n][0], ",".join(f"{a}={b:g}" for a, b in CASES[n][3].items())))
def test_wave_instantiations_match_oracle(need_gpu, n):
    nt, nx, ny, kw = CASES[n]
    d, o, S, Q, Trep = build(n, nt, nx, ny, kw)
    t0, dt = 150.0, 0.1
    for k in range(2):
        t = t0 + (k + 1) * dt
        d.use_bnd_record(0, t - t0, 1.0, Trep)
        d.step(dt, t)
        oracle_step(o, S, Q, Trep, t0, t, dt)
    for f in FIELDS:
        assert np.array_equal(d.get(f), o.get(f), equal_nan=True), f
    a, b = d.cfl(), o.cfl()
    assert a[0] == b[0] and a[1] == pytest.approx(b[1], rel=1e-6)
    d.close()


def test_batched_wave_instantiations_match_oracle(need_gpu):
    """The same domains advancing together."""
    t0 = 150.0
    all_ = [build(n, *c[:3], c[3]) for n, c in enumerate(CASES)]
    ens = Ensemble([a[0] for a in all_], [RunSetup(t0, 0.05, 1e9, t0, 1.0, a[4]) for a in all_])
    for _ in range(2):
        ens.step(1)
        t, dt, steps, status = ens.status()
        assert (status == 0).all()
        for (d, o, S, Q, Trep), tn, dn in zip(all_, t, dt):
            oracle_step(o, S, Q, Trep, t0, tn, dn)
    for n, (d, o, *_) in enumerate(all_):
        for f in FIELDS:
            assert np.array_equal(d.get(f), o.get(f), equal_nan=True), (CASES[n], f)
    ens.close()
    for a in all_:
        a[0].close()
