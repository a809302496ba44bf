"""The slip-rate law of fault creep over both signs of (a-b) sigma and on both
sides of its clamp (|tau / ((a-b) sigma)| = 11): the moment density, the
velocity field and the patches' velocities hold one law."""
import numpy as np
import pytest

import oracle as O
from _cases import oracle_model
from relax_amd import LAYER, PATCH, friction3d, workloads
from relax_amd.model import FAULTCREEP, Model
from test_gpu_creep_bands import check, creep_spec, loaded_state

pytestmark = pytest.mark.gpu

MU = 3e4
ARGS = (1.0, -2.0, 6.0, 10.0, 16.0, 0.3, 0.8, 1.2, 0.2)  # x y z L W strike dip rake beta
RATIOS = (-40.0, -20.0, -15.0, -11.5, -10.5, -5.0, -0.5, -1e-4, 1e-4, 0.5, 5.0, 10.5, 11.5, 15.0)
# FP32 sums of FP64 values: a handful of roundings of 2^-24 each
TOL = 1e-6


def plane_stress(amp):
    """Uniform shear of amp MPa on the plane along its rake."""
    strike, dip, rake = ARGS[5:8]
    n = np.array([np.cos(dip) * np.cos(strike), -np.cos(dip) * np.sin(strike), -np.sin(dip)])
    r = np.array([np.sin(strike) * np.cos(rake) + np.cos(strike) * np.sin(dip) * np.sin(rake),
                  np.cos(strike) * np.cos(rake) - np.sin(strike) * np.sin(dip) * np.sin(rake), np.cos(dip) * np.sin(rake)])
    S = amp * (np.outer(r, n) + np.outer(n, r))
    return np.float32([S[0, 0], S[0, 1], S[0, 2], S[1, 1], S[1, 2], S[2, 2]])


def rel_max(a, b):
    return np.abs(a.astype(np.float64) - b).max() / np.abs(b).max()


@pytest.mark.parametrize("ratio", RATIOS)
def test_rate_law(ratio):
    h3, sx = 16, 32
    st = np.zeros(h3, LAYER)
    st["gammadot0"] = 1e-3
    st["stressexponent"] = 2.0 / ratio  # tau = 2 MPa: no normal traction, no cohesion
    st["friction"] = 0.6
    sig = np.empty((h3, sx, sx, 6), np.float32)
    sig[...] = plane_stress(2.0)
    m, v = np.zeros_like(sig), np.zeros((h3, sx, sx + 2), np.float32)
    rm, rv = m.copy(), v.copy()
    tm = friction3d.frictioneigenstress(*ARGS, sig, MU, st, 0.5, 0.5, 0.5, m, 1e7, v)
    rtm = O.frictioneigenstress(*ARGS, sig, MU, st, 0.5, 0.5, 0.5, rm, 1e7, rv)
    assert np.abs(rm).max() > 0 and np.isfinite(m).all() and np.isfinite(v).all()
    em, ev = rel_max(m, rm), rel_max(v, rv)
    assert em < TOL and ev < TOL
    if ratio > 0:  # a negative rate has no relaxation time
        assert abs(tm / rtm - 1) < TOL
    patch, ref = np.zeros((6, 8), PATCH), np.zeros((6, 8), O.PATCH)
    pargs = ARGS + (2 * h3, 0.5, 0.5, 0.5)
    friction3d.monitorfriction(*pargs, sig, st, patch)
    O.monitorfriction(*pargs, sig.astype(np.float64), st, ref)
    assert np.abs(ref["v"]).max() > 0
    np.testing.assert_allclose(patch["v"], ref["v"], rtol=1e-9, atol=0)


def test_undefined_rate():
    """A locked point where (a-b) sigma is zero: 0/0 is no rate, in the moment
    as in the patches."""
    h3, sx = 16, 32
    st = np.zeros(h3, LAYER)
    st["gammadot0"] = 1e-3
    st["cohesion"] = 10.0
    sig = np.empty((h3, sx, sx, 6), np.float32)
    sig[...] = plane_stress(2.0)
    m = np.zeros_like(sig)
    rm = m.copy()
    friction3d.frictioneigenstress(*ARGS, sig, MU, st, 0.5, 0.5, 0.5, m)
    O.frictioneigenstress(*ARGS, sig, MU, st, 0.5, 0.5, 0.5, rm)
    assert np.isnan(rm).any()
    np.testing.assert_array_equal(np.isnan(m), np.isnan(rm))


@pytest.mark.parametrize("ratio", [-40.0, -15.0, -5.0])
def test_step_with_negative_tauc(ratio):
    """One step of a model whose plane has a negative (a-b) sigma: the fields
    and the patches' rates."""
    s = creep_spec("upright", (64, 64, 64))
    s["friction"] = [(0.0, 1e-6, 3.0 / ratio, 0.0, 0.6, 0.0)]  # tau = 3 MPa in the loaded state
    dt = np.array([1e-2])
    u, tau, sig = loaded_state(s)
    om = oracle_model(s)
    ref = dict(u1=u[0].copy(), u2=u[1].copy(), u3=u[2].copy(), tau=tau.copy(), sig=sig.copy(),
               gamma=np.zeros_like(u[0]), t=0.0, oi=1, i=0)
    O.rk2_run(om, ref, 1, dt)
    t = workloads.tables(s)
    with Model(64, 64, 64, *workloads.spacing(s), *workloads.constants(s), interval=s["interval"]) as m:
        m.set_prestress(t["prestress"])
        m.set_planes(workloads.planes(s))
        m.set_structure(FAULTCREEP, t["friction"])
        m.upload(*u, tau, sig)
        m.run(1, dt_replay=dt)
        out, v = m.download(), m.get_patches()["v"]
    check(out, ref, tau, 64)
    assert (om["patches"]["v"] < 0).any()
    np.testing.assert_allclose(v, om["patches"]["v"], rtol=1e-4, atol=0)
