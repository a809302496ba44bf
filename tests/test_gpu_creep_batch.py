"""A batch of models that all have creeping planes: every member equals its
single run bitwise, the sums of power and C:E^i too, whatever the batch."""
import numpy as np
import pytest

from relax_amd import workloads
from relax_amd.model import Batch

from _cases import small_spec

pytestmark = pytest.mark.gpu

FIELDS = ("u1", "u2", "u3", "tau", "sig", "gamma")
RECORD = ("Dt", "tm", "maxwell", "power", "cei", "t")


def specs(grids):
    return [small_spec("afterslip", sx=n, sx3=n3, seed=k) for k, (n, n3) in enumerate(grids)]


@pytest.mark.parametrize("grids", [((128, 64),) * 3, ((64, 64),) * 2, ((128, 64), (64, 64), (128, 128)),
                                   ((32, 32), (256, 64), (128, 64))], ids=str)
def test_members_equal_their_single_runs(grids):
    nsteps = 3
    alone = []
    for s in specs(grids):
        with workloads.build(s) as m:
            recs = [m.step() for _ in range(nsteps)]
            alone.append((recs, m.download(), m.get_patches()))
    models = [workloads.build(s) for s in specs(grids)]
    with Batch(models) as b:
        for k in range(nsteps):
            recs = b.step()
            for i, r in enumerate(recs):
                for key in RECORD:
                    assert r[key] == alone[i][0][k][key], (i, k, key)
    for m, (_, out, patches) in zip(models, alone):
        got = m.download()
        for key in FIELDS:
            np.testing.assert_array_equal(got[key], out[key], err_msg=key)
        np.testing.assert_array_equal(m.get_patches(), patches)
        m.close()
