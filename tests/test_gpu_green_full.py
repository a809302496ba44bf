"""greenfunctioncowling over the full depth at every depth its column kernels
are compiled for, with body forces above and below the surface; n1/2 + 1
columns leave a ragged last tile.  Both sides transform up to 2^18 points in
FP32: errors of about 18 x 2^-24 each, 4e-6 in all."""
import numpy as np
import pytest

import oracle as O
from _cases import oracle_initial_state, rel_l2, small_spec
from relax_amd import green, workloads

pytestmark = pytest.mark.gpu

LAM, MU, GAM = 3.1e4, 2.8e4, 8.33e-4


@pytest.mark.parametrize("n", [(32, 16, 16), (16, 32, 32), (64, 32, 64), (16, 16, 128), (64, 32, 128), (16, 16, 256),
                               (32, 32, 256), (128, 16, 256), (32, 16, 512), (16, 16, 1024)])
def test_full_depth_solve(n):
    n1, n2, n3 = n
    rng = np.random.default_rng(n1 + n2 + n3)
    c = [np.zeros((n3, n2, n1 + 2), np.float32) for _ in range(3)]
    t = [np.zeros((n2, n1 + 2), np.float32) for _ in range(3)]
    for a in c + t:
        a[..., :n1] = rng.standard_normal(a[..., :n1].shape)
    ref = [a.copy() for a in c + t]
    O.greenfunctioncowling(*ref, 0.9, 1.1, 0.7, LAM, MU, GAM)
    green.greenfunctioncowling(*c, *t, 0.9, 1.1, 0.7, LAM, MU, GAM)
    for a, b in zip(c, ref):
        assert rel_l2(a[..., :n1], b[..., :n1]) < 4e-6


@pytest.mark.parametrize("n", [(32, 32, 512), (64, 128, 512), (128, 32, 512)])
def test_deep_half_columns_match_the_lds_form(n):
    """The register form of 256-deep half columns (with the Nyquist columns,
    the split and the unsplit y order) against the form that keeps them in
    LDS: FP32 rounding of the same transforms, 1e-5 after three steps as for
    the other depths."""
    s = small_spec("powerlaw")
    s.update(sx1=n[0], sx2=n[1], sx3=n[2])
    out = {}
    for v in (0, 3):
        with workloads.build(s) as m:
            m.set_tuning(green=v)
            for _ in range(3):
                m.step(info=False)
            out[v] = m.download()
    for k in ("u1", "u2", "u3"):
        assert rel_l2(out[3][k][..., :n[0]], out[0][k][..., :n[0]]) < 1e-5, k
    for k in ("sig", "tau"):
        assert rel_l2(out[3][k], out[0][k]) < 1e-5, k


@pytest.mark.parametrize("n", [(32, 32, 32), (64, 32, 64), (32, 32, 128), (32, 64, 256), (32, 32, 512)])
def test_cracks_and_point_sources_add_their_upper_half(n):
    """An event with images above the surface solves over the full depth and
    adds the upper half to u, at every depth of the column kernels; the second
    event of the same sources doubles u.  u as for the full-depth solve (4e-6)
    with two roundings of the sum; tau and sig as the set-up's."""
    s = small_spec("powerlaw")
    s.update(sx1=n[0], sx2=n[1], sx3=n[2], tensile=[(1.5e-3, -6.0, 4.0, 1.0, 6.0, 4.0, 30.0, 70.0)],
             mogi=[(4e-3, 8.0, -6.0, 4.0), (-2e-3, -9.0, -9.0, 1.5)])
    st = oracle_initial_state(s)
    with workloads.build(s) as m:
        one = m.download()
        m.event(nyquist=workloads.NYQUIST, **workloads.event_sources(s, 1))
        two = m.download()
    for k in ("u1", "u2", "u3"):
        assert rel_l2(one[k][..., :n[0]], st[k][..., :n[0]]) < 5e-6, k
        assert rel_l2(two[k][..., :n[0]], 2 * st[k][..., :n[0]]) < 5e-6, k
    assert rel_l2(one["tau"], st["tau"]) < 1e-6 and rel_l2(one["sig"], st["sig"]) < 1e-5
