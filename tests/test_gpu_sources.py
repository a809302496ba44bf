"""The source kernels visit only the points that a source of the list can
reach: sources across the grid's seams, on the surface, at the bottom, out of
the grid and wider than it, on grids where a workgroup's points are a part of
a row, several rows or several planes, and lists of more sources than a
workgroup holds at a time.  Fields start at zero, so that a point left out (or
one too many) shows against the oracle."""
import numpy as np
import pytest

import oracle as O
from _cases import rel_l2, small_spec
from relax_amd import elastic3d, workloads
from relax_amd._lib import PLANE
from relax_amd.model import Model

pytestmark = pytest.mark.gpu

LAM, MU, BETA = 2.0e4, 3.0e4, 0.25
GRIDS = {"planes": (16, 16, 16), "rows": (64, 32, 32), "row": (512, 8, 16), "ragged": (48, 22, 20)}
# x, y, z, L, W, strike, dip in samples and radians; the fractions are of the grid
PLACES = {"centre": (0.0, 0.0, 0.2, 5.0, 6.0, 0.4, 0.7), "seam": (0.49, -0.5, 0.1, 4.0, 7.0, 1.9, 0.5),
          "surface": (-0.3, 0.2, 0.0, 3.0, 4.0, -0.6, 0.01), "bottom": (0.1, -0.2, 0.5, 6.0, 3.0, 0.2, 1.1),
          "outside": (0.8, 0.1, 0.1, 3.0, 3.0, 0.3, 0.4), "wide": (0.05, 0.0, 0.1, 60.0, 90.0, 0.8, 0.9)}


def check(pairs):
    """Against the oracle's FP64 geometry rounded once to FP32 (6e-8 of the
    sample): 1e-6 overall, as for single sources elsewhere, and of the largest
    sample at each point."""
    for a, b in pairs:
        assert np.abs(a - b).max() <= 1e-6 * np.abs(b).max()
        assert not b.any() or rel_l2(a, b) < 1e-6


@pytest.mark.parametrize("place", PLACES)
@pytest.mark.parametrize("grid", GRIDS)
def test_each_kernel_reaches_the_oracles_points(grid, place):
    sx1, sx2, sx3 = GRIDS[grid]
    fx, fy, fz, L, W, strike, dip = PLACES[place]
    x, y, z = fx * sx1, fy * sx2, fz * sx3
    plane, d = (x, y, z, L, W, strike, dip), (1.0, 1.0, 1.0)
    new = lambda *s: [np.zeros(s, np.float32) for _ in range(3)]
    f, fo, t, to = (new(sx3, sx2, sx1 + 2), new(sx3, sx2, sx1 + 2), new(sx2, sx1 + 2), new(sx2, sx1 + 2))
    elastic3d.source(MU, 1e-3, *plane, 0.9, BETA, *d, *f, *t)
    O.source(MU, 1e-3, *plane, 0.9, BETA, *d, *fo, *to)
    check(zip(f + t, fo + to))
    f, fo = new(sx3, sx2, sx1 + 2), new(sx3, sx2, sx1 + 2)
    elastic3d.tensilesource(LAM, MU, 1e-3, *plane, BETA, *d, *f)
    O.tensilesource(LAM, MU, 1e-3, *plane, BETA, *d, *fo)
    check(zip(f, fo))
    f, fo = new(sx3, sx2, sx1 + 2), new(sx3, sx2, sx1 + 2)
    elastic3d.mogisource(LAM, MU, 2e-3, x, y, z, *d, *f)
    O.mogisource(LAM, MU, 2e-3, x, y, z, *d, *fo)
    check(zip(f, fo))
    for name, args in (("momentdensityshear", (MU, 1e-3, *plane, 0.9, BETA)),
                       ("momentdensitytensile", (LAM, MU, 1e-3, *plane, BETA)),
                       ("momentdensitymogi", (LAM, MU, 2e-3, x, y, z))):
        s, so = (np.zeros((sx3 // 2, sx2, sx1, 6), np.float32) for _ in range(2))
        getattr(elastic3d, name)(*args, *d, s)
        getattr(O, name)(*args, *d, so)
        check([(s, so)])


@pytest.mark.parametrize("n", [1, 257, 2300])
def test_lists_longer_than_a_workgroups(n):
    """n patches added at once against the oracle's call for each in turn."""
    s = small_spec("maxwell")
    s.update(sx1=64, sx2=32, sx3=32, dx=1.0)
    _, mu, _, beta = workloads.constants(s)
    rng = np.random.default_rng(7)
    p = np.zeros(n, PLANE)
    for name, lo, hi in (("x", -34, 34), ("y", -18, 18), ("z", 0, 16), ("width", 1, 3), ("length", 1, 3),
                         ("strike", 0, 6), ("dip", 0, 1.5), ("rake", -3, 3)):
        p[name] = rng.uniform(lo, hi, n)
    slip = rng.uniform(1e-4, 1e-3, n)
    with Model(s["sx1"], s["sx2"], s["sx3"], *workloads.spacing(s), *workloads.constants(s)) as m:
        m.add_shear(p, slip)
        tau = m.download()["tau"]
    ref = np.zeros_like(tau)
    for q, b in zip(p, slip):
        O.momentdensityshear(mu, b, q["x"], q["y"], q["z"], q["width"], q["length"], q["strike"], q["dip"],
                             q["rake"], beta, *workloads.spacing(s), ref)
    check([(tau, ref)])
