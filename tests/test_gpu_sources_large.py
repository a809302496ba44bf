"""The source kernels' two ways of visiting the points (every point tests the
whole list; a workgroup gathers what its rows can reach) and the gathering's
chunk sizes: large grids whose chunks are a part of a row, several rows or
several planes, against the oracle, and one list by both ways, bitwise."""
import numpy as np
import pytest

import oracle as O
from _cases import small_spec
from relax_amd import SOURCE, elastic3d, workloads
from relax_amd._lib import PLANE
from relax_amd.model import Model
from test_gpu_sources import BETA, LAM, MU, PLACES, check

pytestmark = pytest.mark.gpu

# more than 2^20 points in the top half
GRIDS = {"planes": (8, 16, 16800), "rows": (64, 256, 136), "row": (2048, 8, 132), "ragged": (130, 96, 172)}


@pytest.mark.parametrize("place", PLACES)
@pytest.mark.parametrize("grid", GRIDS)
def test_gathered_sources(grid, place):
    sx1, sx2, sx3 = GRIDS[grid]
    fx, fy, fz, L, W, strike, dip = PLACES[place]
    plane, d = (fx * sx1, fy * sx2, fz * min(sx3, 100), L, W, strike, dip), (1.0, 1.0, 1.0)
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
    elastic3d.mogisource(LAM, MU, 2e-3, *plane[:3], *d, *f)
    O.mogisource(LAM, MU, 2e-3, *plane[:3], *d, *fo)
    check(zip(f, fo))
    for name, args in (("momentdensityshear", (MU, 1e-3, *plane, 0.9, BETA)),
                       ("momentdensitytensile", (LAM, MU, 1e-3, *plane, BETA)),
                       ("momentdensitymogi", (LAM, MU, 2e-3, *plane[:3]))):
        s, so = (np.zeros((sx3 // 2, sx2, sx1, 6), np.float32) for _ in range(2))
        getattr(elastic3d, name)(*args, *d, s)
        getattr(O, name)(*args, *d, so)
        check([(s, so)])


def patches(rng, n, half):
    p = np.zeros(n, SOURCE)
    for name, lo, hi in (("x", -half, half), ("y", -half, half), ("z", 0, half), ("width", 1, 5), ("length", 1, 5),
                         ("strike", 0, 6), ("dip", 0, 1.5), ("rake", -3, 3), ("slip", 1e-4, 1e-3),
                         ("opening", 1e-4, 1e-3)):
        p[name] = rng.uniform(lo, hi, n)
    p["beta"] = BETA
    return p


# the top half of 64x32x32 has 2^15 points: lists of 2^10 go whole, longer ones
# are gathered; over the full depth 2^9
@pytest.mark.parametrize("kind,n", [("sources", 1024), ("tensile", 512), ("tensile", 1024), ("mogi", 512), ("mogi", 1024)])
def test_both_ways_give_the_same_bits(kind, n):
    s = small_spec("maxwell")
    p = patches(np.random.default_rng(5), n + 1, 18)
    p[n]["x"] = 1e6  # reaches nothing
    out = []
    for k in (n, n + 1):
        with Model(64, 32, 32, *workloads.spacing(s), *workloads.constants(s)) as m:
            m.event(**{kind: p[:k]})
            out.append(m.download())
    assert np.abs(out[0]["tau"]).max() > 0 and np.abs(out[0]["u1"]).max() > 0
    for key in ("u1", "u2", "u3", "tau", "sig"):
        np.testing.assert_array_equal(out[0][key], out[1][key], err_msg=key)


def test_chunks_of_several_rows():
    """300 patches over 256x256x128 (chunks of 1024 points: four rows)."""
    s = small_spec("maxwell")
    _, mu, _, beta = workloads.constants(s)
    q = patches(np.random.default_rng(9), 300, 132)
    p = np.zeros(300, PLANE)
    for name in ("x", "y", "z", "width", "length", "strike", "dip", "rake"):
        p[name] = q[name]
    slip = np.ascontiguousarray(q["slip"])
    with Model(256, 256, 128, *workloads.spacing(s), *workloads.constants(s)) as m:
        m.add_shear(p, slip)
        tau = m.download()["tau"]
    ref = np.zeros_like(tau)
    for a, b in zip(p, slip):
        O.momentdensityshear(mu, b, a["x"], a["y"], a["z"], a["width"], a["length"], a["strike"], a["dip"],
                             a["rake"], beta, *workloads.spacing(s), ref)
    check([(tau, ref)])
