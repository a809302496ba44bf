"""grnfct_okada against the oracle where the arc tangents of the four corners
add up to full turns (points close to both sides of the fault), and far away
where the corner terms cancel.  One addition to zero in single precision: the
two agree to a few times 2^-24 of the largest displacement."""
import numpy as np
import pytest

import oracle as O
from relax_amd import okada

pytestmark = pytest.mark.gpu

LAM, MU = 3.2e4, 2.7e4


@pytest.mark.parametrize("dip", [3.0, 30.0, 61.0, 90.0])
@pytest.mark.parametrize("kind", ["strike", "dip", "tensile"])
@pytest.mark.parametrize("dx, size", [(0.37, (4.3, 6.1)), (9.0, (1.0, 1.0))])
def test_near_and_far_field(dip, kind, dx, size):
    n1, n2, n3 = 32, 16, 16
    slip, opening, rake = {"strike": (1e-3, 0.0, 0.0), "dip": (1e-3, 0.0, 90.0), "tensile": (0.0, 1e-3, 0.0)}[kind]
    src = (slip, opening, -1.3, 0.4, 0.6, *size, 23.0, dip, rake)
    ref = [np.zeros((n3, n2, n1 + 2), np.float32) for _ in range(3)]
    O.grnfct_okada(LAM, MU, *src, dx, dx, dx, *ref)
    u = [np.zeros((n3, n2, n1 + 2), np.float32) for _ in range(3)]
    okada.grnfct_okada(LAM, MU, *src, dx, dx, dx, *u)
    top = max(np.abs(b).max() for b in ref)
    for a, b in zip(u, ref):
        assert np.abs(a - b).max() <= 4 * 2.0 ** -24 * top
