"""Surface statistics started between replayed steps: a step captured before
the start holds no statistics kernels, so the start must lead to a new one."""
import numpy as np
import pytest

from caseutil import aerofoil_case
from tandemproject_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [1, 2])
def test_statistics_started_after_a_captured_step(every):
    print("statistics after a captured step, every", every, flush=True)
    lay, ss, p = aerofoil_case(lxibk=(14, 18, 14), letbk=(14, 14), lzebk=(12,))
    got = []
    for graph in (False, True):
        s = api.Solver([(lay, p)])
        for b in range(lay.nb):
            s.set_grid(0, b, ss[b])
        s.setup_geometry()
        s.initialo(0)
        s.step(2, graph=graph)
        s.stats_start(0, every)
        s.step(5, graph=graph)
        s.sync()
        walls = [s.stats_wall(0, b) for b in range(lay.nb)]
        got.append((s.stats_forces(0), walls))
        s.close()
    assert str(got[0][0]) == str(got[1][0]) and "nan" not in str(got[0][0])
    for a, b in zip(got[0][1], got[1][1]):
        assert str(a) == str(b)
