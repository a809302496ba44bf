"""greenfunctioncowling: the traction planes come back as they went in (their
transforms and back), and allocation-free solves on two streams that were
enqueued before either was waited for give what each gives alone."""
import ctypes

import numpy as np
import pytest

import oracle as O
from _cases import rel_l2
from relax_amd import green, load
from test_zz_no_alloc import D2H, GAM, H2D, LAM, MU, _hip, _inputs, _noalloc, _ok

pytestmark = pytest.mark.gpu

DX = (0.9, 1.1, 0.7)


@pytest.mark.parametrize("n", [(32, 16, 16), (64, 32, 64), (16, 16, 128), (128, 16, 256), (32, 16, 512), (16, 16, 1024)])
def test_tractions_come_back(n):
    c, t = _inputs(*n, 7)
    ref = [a.copy() for a in c + t]
    O.greenfunctioncowling(*ref, *DX, LAM, MU, GAM)
    green.greenfunctioncowling(*c, *t, *DX, LAM, MU, GAM)
    # two transforms of up to 2^12 points in FP32: 24 x 2^-24
    for a, b in zip(t, ref[3:]):
        assert rel_l2(a[:, :n[0]], b[:, :n[0]]) < 1.5e-6


@pytest.mark.parametrize("grids", [((128, 128, 128), (128, 128, 128)), ((256, 64, 128), (64, 128, 512)),
                                   ((64, 64, 64), (128, 128, 256))], ids=str)
def test_solves_on_two_streams(grids):
    hip = _hip()
    ins = [[a for part in _inputs(*n, 3 + k) for a in part] for k, n in enumerate(grids)]
    alone = [[a for part in _noalloc(i[:3], i[3:], DX) for a in part] for i in ins]
    streams, dev = [ctypes.c_void_p() for _ in grids], []
    try:
        for s in streams:
            _ok(hip.hipStreamCreate(ctypes.byref(s)))
        for arrays in ins:
            row = []
            dev.append(row)
            for a in arrays:
                d = ctypes.c_void_p()
                _ok(hip.hipMalloc(ctypes.byref(d), a.nbytes))
                row.append(d)
                _ok(hip.hipMemcpy(d, a.ctypes.data, a.nbytes, H2D))
        for n, d, s in zip(grids, dev, streams):
            assert load().relax_greenfunctioncowling_noalloc(*d, *n, *DX, LAM, MU, GAM, s) == 0
        for s in streams:
            _ok(hip.hipStreamSynchronize(s))
        for arrays, row, ref in zip(ins, dev, alone):
            for a, d, r in zip(arrays, row, ref):
                out = np.empty_like(a)
                _ok(hip.hipMemcpy(out.ctypes.data, d, out.nbytes, D2H))
                np.testing.assert_array_equal(out, r)
    finally:
        for row in dev:
            for d in row:
                hip.hipFree(d)
        for s in streams:
            hip.hipStreamDestroy(s)
