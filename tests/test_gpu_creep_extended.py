"""Fault creep together with the extended rheology (weak zones, transient
creep, inter-seismic loading): the points of the creep bands and all others go
to two kernels each, which share the transient strain, the loading and the
minima of five mechanisms.  Every tile kind, single models and batches."""
import numpy as np
import pytest

import oracle as O
from _cases import oracle_model, rel_l2
from relax_amd import workloads
from relax_amd.model import FAULTCREEP, LINEAR, LTRANSIENT, NLTRANSIENT, Batch, Model
from test_gpu_creep_bands import check, creep_spec, loaded_state

pytestmark = pytest.mark.gpu

STEPS = 2


def spec(kind, plane, n):
    s = creep_spec(plane, n)
    s["linear"] = [(9.0, 0.05, 1.0, 0.0, 0.6, 0.0)]
    if kind == "transient":
        s["ltransient"] = [(2.0, 0.4, 1.0, 0.0, 0.6, 1.5e4)]
        s["nltransient"] = [(6.0, 3e7, 3.0, 0.0, 0.6, 2.0e4)]
        s["weak_linear"] = [(0.3, -4.0, -2.0, 4.0, 8.0, 6.0, 5.0, 30.0, 60.0)]
        s["weak_ltransient"] = [(0.8, 3.0, 2.0, 2.0, 6.0, 4.0, 6.0, 0.0, 90.0)]
    else:
        s["inter"] = [(1e-3, -8.0, 2.0, 0.0, 12.0, 5.0, 10.0, 70.0, 30.0)]
        s["inter_tensile"] = [(4e-4, 4.0, 5.0, 2.0, 5.0, 3.0, 0.0, 90.0)]
    return s


def device_model(s):
    m = Model(s["sx1"], s["sx2"], s["sx3"], *workloads.spacing(s), *workloads.constants(s), interval=s["interval"])
    t = workloads.tables(s)
    m.set_prestress(t["prestress"])
    m.set_structure(LINEAR, t["linear"])
    if s.get("ltransient"):
        m.set_structure(LTRANSIENT, t["ltransient"])
        m.set_structure(NLTRANSIENT, t["nltransient"])
    for mech, zones in workloads.weak_zones(s).items():
        m.set_weakzones(mech, zones)
    m.set_planes(workloads.planes(s))
    m.set_structure(FAULTCREEP, t["friction"])
    inter = workloads.interseismic(s)
    if inter is not None:
        m.set_interseismic(*inter)
    u, tau, sig = loaded_state(s)
    m.upload(*u, tau, sig)
    if s.get("ltransient"):
        m.set_transient_strain(np.zeros_like(tau))
    return m


def oracle_steps(s):
    u, tau, sig = loaded_state(s)
    st = dict(u1=u[0], u2=u[1], u3=u[2], tau=tau, sig=sig, gamma=np.zeros_like(u[0]), t=0.0, oi=1, i=0)
    if s.get("ltransient"):
        st["epsilonik"] = np.zeros_like(tau)
    return st, O.rk2_run(oracle_model(s), st, STEPS)


def follow(m, s, ref):
    out = m.download()
    check(out, ref, loaded_state(s)[1], s["sx1"])
    if s.get("ltransient"):
        e, d = ref["epsilonik"], m.transient_strain()
        top = np.abs(e).max()
        assert top > 0 and np.abs(d - e).max() < 1e-4 * top  # every point advanced once
    return out


@pytest.mark.parametrize("kind", ["transient", "loading"])
@pytest.mark.parametrize("plane", ["seam", "flat", "two"])
@pytest.mark.parametrize("n", [(64, 64, 64), (32, 64, 64)])
def test_follows_the_oracle(kind, plane, n):
    s = spec(kind, plane, n)
    ref, info = oracle_steps(s)
    outs = []
    for body in (None, 0, 1) + ((2, 3, 4, 5) if n[0] == 64 else ()):
        with device_model(s) as m:
            if body is not None:
                m.set_tuning(bodyforce=body, green=0, fft_cols=0)
            recs = m.run(STEPS, dt_replay=np.ascontiguousarray(info[:, 0]))
            outs.append(follow(m, s, ref))
        for r, i in zip(recs, info):
            for j, col in enumerate((2, 3, 4, 8, 9)):
                assert abs(r["maxwell"][j] / i[col] - 1) < 1e-5, (body, j)
            assert abs(r["power"] / i[5] - 1) < 1e-4 and abs(r["cei"] / i[6] - 1) < 1e-4
    for o in outs[2:]:  # the tiles give equal results
        for k in ("u1", "u2", "u3", "tau", "sig"):
            np.testing.assert_array_equal(o[k], outs[1][k], err_msg=k)


@pytest.mark.parametrize("grids", [((64, 64, 64),) * 3, ((64, 64, 64), (32, 64, 64), (128, 64, 64))], ids=["one", "mixed"])
def test_batches(grids):
    """A creeping member, an extended one and one that is both: every member
    runs the kernels of both classes."""
    specs = [creep_spec("seam", grids[0]), spec("transient", "flat", grids[1]), spec("loading", "two", grids[2])]
    specs[1].update(planes=None, friction=None)
    refs = []
    for k, s in enumerate(specs):
        if k == 1:  # no plane: the loaded state of the flat one
            s = dict(s, planes=spec("transient", "flat", grids[1])["planes"])
        u, tau, sig = loaded_state(s)
        refs.append(dict(u1=u[0], u2=u[1], u3=u[2], tau=tau, sig=sig, gamma=np.zeros_like(u[0]), t=0.0, oi=1, i=0))
    models, infos = [], []
    for k, (s, st) in enumerate(zip(specs, refs)):
        m = Model(s["sx1"], s["sx2"], s["sx3"], *workloads.spacing(s), *workloads.constants(s), interval=s["interval"])
        t = workloads.tables(s)
        m.set_prestress(t["prestress"])
        m.set_structure(LINEAR, t["linear"])
        if s.get("ltransient"):
            st["epsilonik"] = np.zeros_like(st["tau"])
            m.set_structure(LTRANSIENT, t["ltransient"])
            m.set_structure(NLTRANSIENT, t["nltransient"])
        for mech, zones in workloads.weak_zones(s).items():
            m.set_weakzones(mech, zones)
        if s["planes"]:
            m.set_planes(workloads.planes(s))
            m.set_structure(FAULTCREEP, t["friction"])
        if s.get("inter"):
            m.set_interseismic(*workloads.interseismic(s))
        m.upload(st["u1"], st["u2"], st["u3"], st["tau"], st["sig"])
        if s.get("ltransient"):
            m.set_transient_strain(st["epsilonik"])
        models.append(m)
        infos.append(O.rk2_run(oracle_model(s), st, STEPS))
    with Batch(models) as b:
        for k in range(STEPS):
            for r, info in zip(b.step(), infos):
                assert abs(r["Dt"] / info[k, 0] - 1) < 1e-5 and abs(r["power"] / info[k, 5] - 1) < 1e-4
    for m, s, st in zip(models, specs, refs):
        out = m.download()
        for key in ("u1", "u2", "u3"):
            assert rel_l2(out[key][..., :s["sx1"]], st[key][..., :s["sx1"]]) < 1e-4, key
        for key in ("tau", "sig"):
            assert rel_l2(out[key], st[key]) < 1e-4, key
        if s.get("ltransient"):
            e = st["epsilonik"]
            assert np.abs(m.transient_strain() - e).max() < 1e-4 * np.abs(e).max()
        m.close()
