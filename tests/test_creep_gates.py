"""The points that the creep kernels take (rheology.h: in_band, column_band,
band_box), compiled for the host: every point that passes the gates of
frictioneigenstress lies in the band, its column's depth range and the box of
the band launches, on the gates' very edges too, and no geometry makes a box
that is not on the grid."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from relax_amd import PLANE
from relax_amd import build as hipbuild
from relax_amd._lib import ptr

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BETA = 0.2


@pytest.fixture(scope="module")
def native(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("creep_gates") / "creep_gates.so")
    lib = os.path.join(ROOT, "relax_amd")
    cmd = [hipbuild.HIPCC, "-x", "hip", "--offload-arch=gfx950", "--cuda-host-only", "-O2", "-std=c++17", "-fPIC", "-mfma",
           "-shared", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(lib, "csrc"),
           os.path.join(ROOT, "tests", "native", "creep_gates.cpp"), "-o", so,
           "-L" + lib, "-l:librelax_hip.so", "-Wl,-rpath," + lib]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    native = ctypes.CDLL(so)
    for fn in (native.creep_box, native.creep_sweep):
        fn.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_double] + [ctypes.c_void_p] * 3
    return native


def plane(x, y, z, length, width, strike, dip, rake=0.0):
    p = np.zeros(1, PLANE)
    p[0] = (x, y, z, width, length, strike, dip, rake, 1, 1)
    return p


def call(fn, planes, n, dx, nout, dtype):
    planes = np.ascontiguousarray(planes)
    n, dx, out = np.array(n, np.int32), np.array(dx, np.float64), np.zeros(nout, dtype)
    fn(ptr(planes), len(planes), BETA, ptr(n), ptr(dx), ptr(out))
    return out


NAN, INF = float("nan"), float("inf")


@pytest.mark.parametrize("geometry", [
    dict(x=NAN), dict(y=NAN), dict(z=NAN), dict(length=NAN), dict(width=NAN), dict(length=NAN, width=NAN), dict(strike=NAN),
    dict(x=INF), dict(y=-INF), dict(z=INF), dict(length=INF), dict(x=INF, width=INF), dict(x=1e300), dict(x=-1e12),
    dict(length=-20.0, width=-30.0), dict(length=-20.0), dict(width=-20.0), dict(length=0.0, width=0.0)], ids=str)
@pytest.mark.parametrize("pair", [False, True])
def test_box_is_on_the_grid(native, geometry, pair):
    n = (64, 32, 16)
    p = plane(**{**dict(x=1.0, y=2.0, z=3.0, length=8.0, width=6.0, strike=0.4, dip=0.7), **geometry})
    if pair:
        p = np.concatenate([p, plane(-5.0, 1.0, 2.0, 8.0, 6.0, 0.1, 0.3)])
    zmax, x0, nx, y0, ny = call(native.creep_box, p, n, (1.0, 1.0, 1.0), 5, np.int32)
    assert 0 <= zmax <= n[2] and 0 <= x0 < n[0] and 1 <= nx <= n[0] and 0 <= y0 < n[1] and 1 <= ny <= n[1]
    _, _, _, outside, columns = call(native.creep_sweep, p, n, (1.0, 1.0, 1.0), 5, np.int64)
    assert (outside, columns) == (0, 0)


def edge_planes(rng, dx):
    """Planes whose gates pass through grid points: centre and extent in whole
    or half samples of decimal spacings, dips and strikes of round degrees."""
    out = []
    for _ in range(int(rng.integers(1, 3))):
        half = lambda a, b: 0.5 * int(rng.integers(2 * a, 2 * b))
        length, width = half(2, 20), half(2, 20)
        # z + Lp, x + wl on whole samples: (1 + 2 beta)/2 = 0.7 of the extent
        grow = rng.integers(2) * 0.7
        z = half(0, 12) + (grow * length if rng.integers(2) else 0.0)
        x, y = half(-16, 16) + grow * max(length, width), half(-8, 8) - grow * max(length, width)
        strike, dip = np.deg2rad(15.0 * rng.integers(0, 24)), np.deg2rad(15.0 * rng.integers(-6, 13))
        out.append(plane(x * dx[0], y * dx[1], z * dx[2], length * dx[2], width * dx[2], strike, dip))
    return np.concatenate(out)


@pytest.mark.parametrize("dx", [(0.1, 0.1, 0.1), (0.3, 0.7, 0.1), (1.0, 1.0, 1.0), (1e3 / 3, 1e3 / 3, 50.0), (0.05, 0.6, 0.9)])
@pytest.mark.parametrize("n", [(64, 32, 16), (32, 32, 32)])
def test_points_on_the_gates(native, n, dx):
    rng = np.random.default_rng(11)
    total = np.zeros(5, np.int64)
    for _ in range(250):
        total += call(native.creep_sweep, edge_planes(rng, dx), n, dx, 5, np.int64)
    assert total[0] > 10000
    assert (total[1:] == 0).all(), total
