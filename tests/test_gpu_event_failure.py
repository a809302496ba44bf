"""An event that fails leaves the model's state as it was.  The failure is a
HIP error left pending by a call of the caller's own (an invalid device
number), which the library's first launch check reports."""
import ctypes

import numpy as np
import pytest

from relax_amd import RelaxError, workloads

from _cases import small_spec

pytestmark = pytest.mark.gpu

KEYS = ("u1", "u2", "u3", "tau", "sig", "gamma")


def test_failed_event_keeps_the_state():
    s = small_spec("maxwell", sx=32, sx3=32)
    s.update(tensile=[(1e-3, -3.0, 0.0, 2.0, 6.0, 5.0, 30.0, 80.0)], mogi=[(1e-3, 2.0, 1.0, 5.0)], deck=[])
    event = workloads.event_sources(s, 1)
    with workloads.build(s) as m:
        hip = ctypes.CDLL("libamdhip64.so.7")  # as loaded with the library
        m.step()
        before = m.download()
        assert np.abs(before["sig"]).max() > 0
        hip.hipGetLastError()
        assert hip.hipSetDevice(9999) != 0
        with pytest.raises(RelaxError):
            m.event(**event)
        after = m.download()
        for k in KEYS:
            np.testing.assert_array_equal(after[k], before[k], err_msg=k)
        # the error is reported once: the same event then goes through
        m.event(**event)
        again = m.download()
    assert rel(again["sig"], before["sig"]) > 1e-3


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)
