"""Fault creep is computed by kernels of its own in the bands of the creeping
planes and by none elsewhere: planes that cross the grid's seams, reach the
surface or the bottom, lie flat or stand upright, overlap or cover the grid,
on grids of every tile kind, alone and in batches.  The stress is uniform and
loads every plane along its rake, so that each point of a band creeps and a
point or tile that is left out shows in the oracle's increments."""
import numpy as np
import pytest

import oracle as O
from _cases import oracle_model, rel_l2, small_spec
from relax_amd import workloads
from relax_amd.model import FAULTCREEP, LINEAR, POWERLAW, Batch, Model

pytestmark = pytest.mark.gpu

PLANES = {
    "seam": [dict(x=20.0, y=26.0, z=2.0, length=22.0, width=8.0, strike=35.0, dip=40.0, rake=90.0)],
    "upright": [dict(x=-9.0, y=-6.5, z=0.0, length=18.0, width=9.0, strike=60.0, dip=90.0, rake=0.0)],
    "flat": [dict(x=-8.0, y=6.0, z=6.4, length=14.0, width=12.0, strike=0.0, dip=4.0, rake=-90.0)],
    "bottom": [dict(x=-5.0, y=0.0, z=24.0, length=9.0, width=8.0, strike=15.0, dip=50.0, rake=45.0)],
    "two": [dict(x=-22.0, y=-20.0, z=1.0, length=7.0, width=5.0, strike=0.0, dip=30.0, rake=-90.0),
            dict(x=9.0, y=17.0, z=12.0, length=9.0, width=6.0, strike=0.0, dip=30.0, rake=-90.0)],
    "wide": [dict(x=-30.0, y=18.0, z=0.5, length=60.0, width=40.0, strike=5.0, dip=35.0, rake=-90.0)],
}


def creep_spec(name, n):
    s = small_spec("afterslip")
    s.update(sx1=n[0], sx2=n[1], sx3=n[2], nonlinear=None, deck=[], planes=PLANES[name])
    return s


def loaded_state(s):
    """u = 0, tau = -S, sig = S, with S = 3 MPa of shear on the first plane
    along its rake."""
    p = workloads.planes(s)[0]
    cs, ss, cd, sd = np.cos(p["strike"]), np.sin(p["strike"]), np.cos(p["dip"]), np.sin(p["dip"])
    cr, sr = np.cos(p["rake"]), np.sin(p["rake"])
    n = np.array([cd * cs, -cd * ss, -sd])
    r = np.array([ss * cr + cs * sd * sr, cs * cr - ss * sd * sr, cd * sr])
    S = 3.0 * (np.outer(n, r) + np.outer(r, n))
    shape = (s["sx3"] // 2, s["sx2"], s["sx1"])
    sig = np.empty(shape + (6,), np.float32)
    sig[...] = S[[0, 0, 0, 1, 1, 2], [0, 1, 2, 1, 2, 2]]
    u = [np.zeros(shape[:2] + (shape[2] + 2,), np.float32) for _ in range(3)]
    return u, -sig, sig


def device_model(s):
    dx = workloads.spacing(s)
    m = Model(s["sx1"], s["sx2"], s["sx3"], *dx, *workloads.constants(s), interval=s["interval"])
    t = workloads.tables(s)
    m.set_prestress(t["prestress"])
    m.set_structure(LINEAR, None)
    m.set_structure(POWERLAW, t["nonlinear"])
    m.set_planes(workloads.planes(s))
    m.set_structure(FAULTCREEP, t["friction"])
    u, tau, sig = loaded_state(s)
    m.upload(*u, tau, sig)
    return m


def oracle_step(s):
    u, tau, sig = loaded_state(s)
    st = dict(u1=u[0], u2=u[1], u3=u[2], tau=tau, sig=sig, gamma=np.zeros_like(u[0]), t=0.0, oi=1, i=0)
    info = O.rk2_run(oracle_model(s), st, 1)
    return st, info[:, 0]


def check(out, ref, tau0, n1):
    d, e = out["tau"] - tau0, ref["tau"] - tau0
    assert np.abs(e).max() > 0
    # every point's increment follows the oracle
    assert np.abs(np.abs(d).max(-1) - np.abs(e).max(-1)).max() < 1e-4 * np.abs(e).max()
    assert rel_l2(d, e) < 1e-4
    for k in ("u1", "u2", "u3"):
        assert rel_l2(out[k][..., :n1], ref[k][..., :n1]) < 1e-4, k
    assert rel_l2(out["sig"], ref["sig"]) < 1e-4


@pytest.mark.parametrize("name", sorted(PLANES))
@pytest.mark.parametrize("n", [(64, 64, 64), (32, 64, 64), (128, 64, 64)])
def test_creep_follows_the_oracle(name, n):
    s = creep_spec(name, n)
    ref, dt = oracle_step(s)
    tau0 = loaded_state(s)[1]
    outs = []
    for body in (None, 1) + ((4, 5) if n[0] == 64 else ()):
        with device_model(s) as m:
            if body is not None:
                m.set_tuning(bodyforce=body)
            m.run(1, dt_replay=dt)
            outs.append(m.download())
        check(outs[-1], ref, tau0, n[0])


def test_batches_of_creeping_planes():
    specs = [creep_spec("seam", (64, 64, 64)), creep_spec("two", (64, 64, 64)), creep_spec("wide", (64, 64, 64))]
    mixed = specs + [creep_spec("flat", (32, 64, 64)), creep_spec("upright", (128, 64, 64))]
    for group in (specs, mixed):
        models = [device_model(s) for s in group]
        with Batch(models) as b:
            recs = b.step()
            for s, m, r in zip(group, models, recs):
                ref, dt = oracle_step(s)
                assert abs(r["Dt"] / dt[0] - 1) < 1e-5
                check(m.download(), ref, loaded_state(s)[1], s["sx1"])
        for m in models:
            m.close()
